// Batched GPU encoder of the fp8 exponent Huffman row format
// (encode, codec.py:125-198), producing the bytes of the host encoder
// (codec_host.cpp) and of the reference.
//
// The plan: encode_hist_kernel and encode_words_kernel (chunks of 512 values
// and more: encode_count_kernel and encode_sizes_kernel), several workgroups
// per row; or encode_plan_kernel, one per row, for C callers of xp_encode_rows,
// which has no workspace (the Python package always gives one):
//   1. exponent histogram: per-thread counters in LDS, then summed;
//   2. the code by one wave, the 512-entry LUT by the workgroup;
//   3. Huffman words per chunk: the decoder loads a word before symbol i
//      whenever fewer than LIMIT bits are left, so a chunk whose last symbol
//      starts at bit b needs (b + LIMIT - 1) / 32 + 1 words; summed per
//      group and scanned into gstart, written to the record's header.
// encode_groups_kernel, one workgroup per 8 groups of a row (per 2 where the
// groups are few, see kSegments):
//   4. the code again, from the row's LUT (every symbol has a code of at
//      most LIMIT bits, so each one appears in the 9-bit table with its
//      length, and the canonical codes follow from the lengths); then each
//      32-lane half-wave encodes one group: its lanes walk their chunks
//      in lockstep, two symbols at a time, run the decoder's refill rule, and
//      give each word the (symbol index, lane) rank of its refill -- the wave
//      ballot's count of refilling lanes below, as the decoder computes it. A
//      lane emits a word once its 32 bits are complete. The lane also writes
//      its sign/mantissa nibble words.
// The record is written whole: nibbles and Huffman words by the groups
// launch, gstart and the zero tail up to the pitch by it or by
// encode_plan_kernel. A row that does not fit its pitch writes nothing but its
// LUT and needed bytes.
#include "code_build.h"
#include "common.h"

namespace xp {
namespace {

constexpr int kThreads = 256;
constexpr int kMaxGroups = 4096;  // groups per row a workgroup scans in LDS
constexpr int kGroupsPerBlock = 2 * kThreads / 64;  // 8: one per half-wave
// The plan's two passes over a row run in one workgroup per row: 16 waves,
// each lane with four 16-byte loads in flight, so that a pass is not a
// chain of load latencies.
constexpr int kPlanThreads = 1024;
constexpr int kPlanUnroll = 4;

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4_any __attribute__((ext_vector_type(4), aligned(4)));

struct EncodeArgs {
  const uint8_t* raw;
  int64_t raw_stride;  // bytes between rows of raw
  int64_t n;           // values per row
  int chunk;           // values per lane chunk (a power of two, 16..1024)
  int G;               // groups per row
  uint8_t* rec;
  int64_t pitch;       // bytes between records, the record size
  uint8_t* lut;
  int64_t lut_stride;  // bytes between LUTs
  int64_t* needed;     // record bytes each row needs
  uint32_t* hist;      // split plan: [row][part][16] exponent counts
  int32_t* words;      // split plan: [row][G] Huffman words per group
  int parts;           // split plan: parts of a row's histogram
  uint32_t* counts;    // split plan, long chunks: [row][chunk][8] (see encode_count_kernel)
};

// A row's code, built by one wave and the same in every lane of it: lane l
// stands for symbol l & 15, whose count it gives and whose code length and
// code it gets. The lengths are code::code_lengths', whose selection of the
// lightest node over (count, id) is a merge of two queues: the symbols sorted
// by (count, symbol), and the merged nodes, which appear in ascending (count,
// id) order because counts only grow; on equal counts the symbol goes first,
// as its id is lower. Queue entries live in lane registers (readlane and
// writelane at wave-uniform indices), so nothing goes through LDS. One thread
// selecting over 16 nodes, and a LUT looked up entry by entry, were a large
// part of the 266 us that the plan of one 2 MiB row took.
__device__ __forceinline__ double lane_double(double v, int lane) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                          __builtin_amdgcn_readlane(__double2loint(v), lane));
}

__device__ __forceinline__ int wave_lengths(double count) {
  const int lane = threadIdx.x & 63, sym = lane & 15;
  // Place in the sorted order, then sorted counts and symbols by lane.
  int rank = 0;
#pragma unroll
  for (int t = 0; t < code::kSyms; ++t) {
    const double c = lane_double(count, t);
    rank += c < count || (c == count && t < sym) ? 1 : 0;
  }
  // Queue ends read as infinity: leaves past lane 15, nodes not yet merged.
  const int to = 4 * ((lane & ~15) + rank);
  const int inf_hi = 0x7ff00000;
  int leaf_lo = __builtin_amdgcn_ds_permute(to, __double2loint(count));
  int leaf_hi = __builtin_amdgcn_ds_permute(to, __double2hiint(count));
  const int leaf_bit = __builtin_amdgcn_ds_permute(to, 1 << sym);
  leaf_lo = lane < code::kSyms ? leaf_lo : 0;
  leaf_hi = lane < code::kSyms ? leaf_hi : inf_hi;
  int node_lo = 0, node_hi = inf_hi, node_members = 0;  // merged node i in lane i
  int length = 0;
  int leaf = 0, head = 0;
  auto pair_double = [](int hi, int lo, int at) {
    return __hiloint2double(__builtin_amdgcn_readlane(hi, at), __builtin_amdgcn_readlane(lo, at));
  };
  for (int step = 0; step < code::kSyms - 1; ++step) {
    // The two lightest of the queues' first two entries each.
    const double l0 = pair_double(leaf_hi, leaf_lo, leaf), l1 = pair_double(leaf_hi, leaf_lo, leaf + 1);
    const double n0 = pair_double(node_hi, node_lo, head), n1 = pair_double(node_hi, node_lo, head + 1);
    const int bl0 = __builtin_amdgcn_readlane(leaf_bit, leaf), bl1 = __builtin_amdgcn_readlane(leaf_bit, leaf + 1);
    const int bn0 = __builtin_amdgcn_readlane(node_members, head);
    const int bn1 = __builtin_amdgcn_readlane(node_members, head + 1);
    const int leaves = __builtin_amdgcn_readfirstlane(l1 <= n0 ? 2 : (n1 < l0 ? 0 : 1));
    const double sum = (leaves > 0 ? l0 : n1) + (leaves == 2 ? l1 : n0);
    const int members = (leaves > 0 ? bl0 : bn1) | (leaves == 2 ? bl1 : bn0);
    leaf += leaves;
    head += 2 - leaves;
    length += (members >> sym) & 1;
    node_lo = lane == step ? __double2loint(sum) : node_lo;
    node_hi = lane == step ? __double2hiint(sum) : node_hi;
    node_members = lane == step ? members : node_members;
  }
  return length;
}

__device__ __forceinline__ int wave_code_lengths(uint32_t hist) {
  double count = static_cast<double>(hist > 1 ? hist : 1);
  for (int k = 0;; ++k) {
    if (k > 0) {  // as code::code_lengths: k never passes LIMIT
      double sum = 0.0;
#pragma unroll
      for (int i = 0; i < code::kSyms; ++i) sum += lane_double(count, i);
      const double floor_c = sum / static_cast<double>(1 << (XP_LIMIT - k));
      count = count > floor_c ? count : floor_c;
    }
    const int length = wave_lengths(count);
    if (!__builtin_amdgcn_ballot_w64(length > XP_LIMIT)) return length;
  }
}

// code::canonical_codes of lane l's symbol l & 15.
__device__ __forceinline__ int wave_canonical_code(int length) {
  const int lane = threadIdx.x & 63, sym = lane & 15;
  uint32_t first = 0, code = 0, prev = 0, below = 0;
#pragma unroll
  for (int L = 1; L <= XP_LIMIT; ++L) {
    const uint32_t of = static_cast<uint32_t>(__builtin_amdgcn_ballot_w64(length == L)) & 0xffffu;
    code = (code + prev) << 1;
    prev = static_cast<uint32_t>(__popc(of));
    if (length == L) {
      first = code;
      below = static_cast<uint32_t>(__popc(of & ((1u << sym) - 1u)));
    }
  }
  return static_cast<int>(__brev(first + below) >> (32 - length));
}

// Lengths of the four bytes of w as a sum. lb[k] holds the code lengths of
// symbols 4k..4k+3 as bytes. Each byte's symbol (its exponent field) selects
// its length with byte permutes: one over symbols 0-7, one over 8-15, and a
// third that takes each byte from the one its symbol's bit 3 names; a sum
// of absolute byte differences against zero adds the four lengths.
__device__ __forceinline__ uint32_t sum_lengths4(uint32_t w, const uint32_t (&lb)[4]) {
  const uint32_t sym = (w >> 3) & 0x0f0f0f0fu;
  const uint32_t low = sym & 0x07070707u;
  const uint32_t a = __builtin_amdgcn_perm(lb[1], lb[0], low);  // symbols 0-7
  const uint32_t b = __builtin_amdgcn_perm(lb[3], lb[2], low);  // symbols 8-15
  const uint32_t pick = ((sym >> 1) & 0x04040404u) | 0x03020100u;  // byte i of a, or of b for symbols 8-15
  return __builtin_amdgcn_sad_u8(__builtin_amdgcn_perm(b, a, pick), 0u, 0u);
}

// The code lengths as bytes, symbol s in byte s % 4 of lb[s / 4].
__device__ __forceinline__ void pack_lengths(const int32_t* s_len, uint32_t (&lb)[4]) {
#pragma unroll
  for (int k = 0; k < 4; ++k) lb[k] = 0u;
#pragma unroll
  for (int s = 0; s < code::kSyms; ++s) lb[s / 4] |= static_cast<uint32_t>(s_len[s]) << (8 * (s % 4));
}

// Words per chunk: (start bit of its last symbol + LIMIT - 1) / 32 + 1. A
// thread holds the 16 values at offset off of the row; a chunk's pieces are
// spread over consecutive threads, so each chunk is summed by a power-of-two
// set of `per` = chunk / 16 lanes of one wave (at most 64), and its last lane
// adds the chunk's words to its group's.
__device__ __forceinline__ void add_chunk_words(const u32x4& v, int64_t off, int chunk, int per,
                                                const uint32_t (&lb)[4], int32_t* s_words, int64_t g_base) {
  uint32_t bits = sum_lengths4(v.x, lb) + sum_lengths4(v.y, lb) + sum_lengths4(v.z, lb) + sum_lengths4(v.w, lb);
  const bool last = ((off + 16) % chunk) == 0;
  if (last) {  // not the last symbol
    const uint32_t s3 = v.w >> 27 & 15u;
    const bool hi = s3 >= 8u;
    bits -= __builtin_amdgcn_perm(hi ? lb[3] : lb[1], hi ? lb[2] : lb[0], (s3 & 7u) | 0x0c0c0c00u);
  }
  for (int d = 1; d < per; d <<= 1) bits += __shfl_xor(bits, d, per);
  if (last)
    atomicAdd(&s_words[off / (int64_t(chunk) * XP_LANES) - g_base],
              static_cast<int32_t>((bits + XP_LIMIT - 1) / 32 + 1));
}

// The LUT from the lengths and codes, by a whole workgroup: a sixteenth of the
// threads per symbol, which owns the windows whose low bits are its code.
__device__ __forceinline__ void write_lut(const int32_t* s_len, const int32_t* s_code, uint8_t* lut, int threads) {
  const int per = threads / code::kSyms, sym = threadIdx.x / per;
  const int n = s_len[sym], code = s_code[sym];
  for (int i = threadIdx.x % per; i < XP_LUT_BYTES >> n; i += per)
    lut[code | (i << n)] = static_cast<uint8_t>((sym << 4) | n);
}

// ---- the plan of a row by several workgroups ----
//
// With a workspace the plan's two passes are launches of their own over
// parts of the rows, so that a few rows fill the GPU and many rows leave no
// partly empty round of one workgroup per row. One 2 MiB row: 266 us in one
// workgroup, 7 + 12 us here; 256 rows: 316 us, 119 + 143 us (537 MB read
// twice, at 4.5 and 3.8 TB/s; half of what was saved is the code's). Long
// chunks are read once, see encode_count_kernel.

// Exponent counts of part `blockIdx.x % parts` (kPartBytes values) of a row.
// Each thread counts into its own LDS counters with atomic adds whose result
// is not returned (see encode_plan_kernel).
constexpr int64_t kPartBytes = 1 << 16;

__global__ void __launch_bounds__(kThreads) encode_hist_kernel(EncodeArgs a) {
  __shared__ uint32_t s_hist[code::kSyms][kThreads];
  const int row = blockIdx.x / a.parts, part = blockIdx.x % a.parts;
  const int tid = threadIdx.x;
  const uint8_t* raw = a.raw + static_cast<int64_t>(row) * a.raw_stride;
  const int64_t lo = part * kPartBytes, hi = lo + kPartBytes < a.n ? lo + kPartBytes : a.n;
  constexpr int64_t kStep = int64_t(kThreads) * 16;
  u32x4 v[kPlanUnroll];
#pragma unroll
  for (int u = 0; u < kPlanUnroll; ++u)
    if (lo + tid * 16 + u * kStep < hi) v[u] = *reinterpret_cast<const u32x4*>(raw + lo + tid * 16 + u * kStep);
  for (int s = 0; s < code::kSyms; ++s) s_hist[s][tid] = 0;
  for (int64_t off0 = lo + tid * 16; off0 < hi; off0 += kStep * kPlanUnroll) {
#pragma unroll
    for (int u = 0; u < kPlanUnroll; ++u) {
      if (off0 + u * kStep >= hi) continue;
      const u32x4 x = v[u];
      const int64_t next = off0 + (u + kPlanUnroll) * kStep;
      if (next < hi) v[u] = *reinterpret_cast<const u32x4*>(raw + next);
      const uint32_t w[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int b = 0; b < 4; ++b) atomicAdd(&s_hist[(w[k] >> (8 * b + 3)) & 15u][tid], 1u);
    }
  }
  __syncthreads();
  // 16 threads per symbol, 16 counters each.
  const int sym = tid >> 4, at = tid & 15;
  uint32_t t = 0;
#pragma unroll
  for (int i = 0; i < kThreads / 16; ++i) t += s_hist[sym][at + 16 * i];
#pragma unroll
  for (int d = 8; d >= 1; d >>= 1) t += __shfl_xor(t, d, 16);
  if (at == 0) a.hist[static_cast<int64_t>(blockIdx.x) * code::kSyms + sym] = t;
}

// The row's code from its parts' counts, by the first wave of a workgroup.
__device__ __forceinline__ void wave_row_code(const EncodeArgs& a, int row, int32_t* s_len, int32_t* s_code) {
  const int tid = threadIdx.x;
  const uint32_t* h = a.hist + static_cast<int64_t>(row) * a.parts * code::kSyms + (tid & 15);
  uint32_t t = 0;
#pragma unroll 4
  for (int i = tid >> 4; i < a.parts; i += 4) t += h[i * code::kSyms];
  t += __shfl_xor(t, 16, 64);
  t += __shfl_xor(t, 32, 64);
  const int length = wave_code_lengths(t);
  const int code = wave_canonical_code(length);
  if (tid < code::kSyms) {
    s_len[tid] = length;
    s_code[tid] = code;
  }
}

// The row's code (each workgroup for itself; the
// row's first one writes the LUT), then the Huffman words of `groups` groups
// (1 to 8: as few as leave the launch within kWordsBlocks workgroups, so that
// a row's code is not built many more times than there are groups in flight).
constexpr int64_t kWordsBlocks = 2048;

__global__ void __launch_bounds__(kThreads) encode_words_kernel(EncodeArgs a, int groups, int blocks_per_row) {
  __shared__ int32_t s_len[code::kSyms];
  __shared__ int32_t s_code[code::kSyms];
  __shared__ int32_t s_words[kGroupsPerBlock];
  const int row = blockIdx.x / blocks_per_row, part = blockIdx.x % blocks_per_row;
  const int tid = threadIdx.x;
  const uint8_t* raw = a.raw + static_cast<int64_t>(row) * a.raw_stride;
  const int64_t group = int64_t(a.chunk) * XP_LANES;
  const int64_t g0 = int64_t(part) * groups;
  const int64_t lo = g0 * group, end = lo + groups * group, hi = end < a.n ? end : a.n;
  constexpr int64_t kStep = int64_t(kThreads) * 16;
  u32x4 v[kPlanUnroll];
#pragma unroll
  for (int u = 0; u < kPlanUnroll; ++u)
    if (lo + tid * 16 + u * kStep < hi) v[u] = *reinterpret_cast<const u32x4*>(raw + lo + tid * 16 + u * kStep);
  if (tid < 64) {
    wave_row_code(a, row, s_len, s_code);
  } else if (tid < 64 + kGroupsPerBlock) {
    s_words[tid - 64] = 0;
  }
  __syncthreads();
  if (part == 0) write_lut(s_len, s_code, a.lut + static_cast<int64_t>(row) * a.lut_stride, kThreads);
  uint32_t lb[4];
  pack_lengths(s_len, lb);
  const int per = a.chunk / 16;
  for (int64_t off0 = lo + tid * 16; off0 < hi; off0 += kStep * kPlanUnroll) {
#pragma unroll
    for (int u = 0; u < kPlanUnroll; ++u) {
      const int64_t off = off0 + u * kStep;
      if (off >= hi) continue;
      const u32x4 x = v[u];
      const int64_t next = off + kPlanUnroll * kStep;
      if (next < hi) v[u] = *reinterpret_cast<const u32x4*>(raw + next);
      add_chunk_words(x, off, a.chunk, per, lb, s_words, g0);
    }
  }
  __syncthreads();
  if (tid < groups && g0 + tid < a.G) a.words[static_cast<int64_t>(row) * a.G + g0 + tid] = s_words[tid];
}

// ---- the same for long chunks, whose values are read once ----
//
// A chunk's words follow from its exponent counts and its last symbol, 32
// bytes for 512 values or more, so the histogram launch leaves those (an
// eighth more work: 119 -> 131 us for 256 rows of 2 MiB, 4.3 TB/s) and the
// second launch reads them instead of the row (143 -> 19 us, the code's build
// for most of it). One row: 6 + 12 -> 7 + 9 us. Chunks below 512 values would
// write and read back more than an eighth of the row, and keep the two passes.

constexpr int kCountChunk = 512;  // values per chunk from which a row's chunks are counted

// encode_hist_kernel with each chunk's counts: word s of a chunk holds symbol
// s's count in bits 0-15 and symbol s + 8's in bits 16-27, word 7 the
// chunk's last symbol in bits 28-31. A wave takes 8 chunks at a time, 8 lanes
// each, so that a load covers whole lines; the lanes' counters run on over the
// chunks, and a chunk's counts are what its lanes' sum grew by. Each lane sums
// two symbols, its eight reads rotated by the symbol so that they hit 64 banks.
__global__ void __launch_bounds__(kThreads) encode_count_kernel(EncodeArgs a) {
  __shared__ uint32_t s_hist[code::kSyms][kThreads];
  const int row = blockIdx.x / a.parts, part = blockIdx.x % a.parts;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, c8 = lane >> 3, l8 = lane & 7;
  const int64_t lo = part * kPartBytes, hi = lo + kPartBytes < a.n ? lo + kPartBytes : a.n;
  const int chunk = a.chunk;
  // A row is whole groups of 32 chunks, and a part whole sets of 8.
  const int sets = static_cast<int>((hi - lo) / (8 * chunk));
  const uint8_t* src = a.raw + static_cast<int64_t>(row) * a.raw_stride + lo + c8 * chunk + 16 * l8;
  uint32_t* out = a.counts + (static_cast<int64_t>(row) * (a.n / chunk) + lo / chunk) * 8;
  u32x4 v[4];
  auto request = [&](int set, int at) {
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = *reinterpret_cast<const u32x4*>(src + int64_t(set) * 8 * chunk + at + 128 * k);
  };
  if (wave < sets) request(wave, 0);
  for (int s = 0; s < code::kSyms; ++s) s_hist[s][tid] = 0;
  uint32_t below0 = 0, below1 = 0;  // the sums after the set before
  for (int set = wave; set < sets; set += kThreads / 64) {
    uint32_t last = 0;
    for (int at = 0; at < chunk; at += kCountChunk) {
      u32x4 x[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) x[k] = v[k];
      if (at + kCountChunk < chunk)
        request(set, at + kCountChunk);
      else if (set + kThreads / 64 < sets)
        request(set + kThreads / 64, 0);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint32_t w[4] = {x[k].x, x[k].y, x[k].z, x[k].w};
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int b = 0; b < 4; ++b) atomicAdd(&s_hist[(w[i] >> (8 * b + 3)) & 15u][tid], 1u);
      }
      last = x[3].w >> 27 & 15u;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    uint32_t sum0 = 0, sum1 = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int at = (tid & ~7) + ((i + l8) & 7);
      sum0 += s_hist[l8][at];
      sum1 += s_hist[l8 + 8][at];
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const uint32_t n0 = sum0 - below0, n1 = sum1 - below1;
    below0 = sum0;
    below1 = sum1;
    out[(int64_t(set) * 8 + c8) * 8 + l8] = n0 | n1 << 16 | (l8 == 7 ? last << 28 : 0u);
  }
  __syncthreads();
  const int sym = tid >> 4, at = tid & 15;
  uint32_t t = 0;
#pragma unroll
  for (int i = 0; i < kThreads / 16; ++i) t += s_hist[sym][at + 16 * i];
#pragma unroll
  for (int d = 8; d >= 1; d >>= 1) t += __shfl_xor(t, d, 16);
  if (at == 0) a.hist[static_cast<int64_t>(blockIdx.x) * code::kSyms + sym] = t;
}

// encode_words_kernel from the chunks' counts, a thread per chunk, `groups`
// (a multiple of 8) groups per workgroup.
__global__ void __launch_bounds__(kThreads) encode_sizes_kernel(EncodeArgs a, int groups, int blocks_per_row) {
  __shared__ int32_t s_len[code::kSyms];
  __shared__ int32_t s_code[code::kSyms];
  const int row = blockIdx.x / blocks_per_row, part = blockIdx.x % blocks_per_row;
  const int tid = threadIdx.x;
  const int g0 = part * groups, g1 = g0 + groups < a.G ? g0 + groups : a.G;
  const uint32_t* counts = a.counts + static_cast<int64_t>(row) * (a.n / a.chunk) * 8;
  int c = g0 * XP_LANES + tid;
  u32x4 lo = {0, 0, 0, 0}, hi = {0, 0, 0, 0};
  if (c < g1 * XP_LANES) {
    lo = *reinterpret_cast<const u32x4_any*>(counts + int64_t(c) * 8);
    hi = *reinterpret_cast<const u32x4_any*>(counts + int64_t(c) * 8 + 4);
  }
  if (tid < 64) wave_row_code(a, row, s_len, s_code);
  __syncthreads();
  if (part == 0) write_lut(s_len, s_code, a.lut + static_cast<int64_t>(row) * a.lut_stride, kThreads);
  uint32_t len[code::kSyms];
#pragma unroll
  for (int s = 0; s < code::kSyms; ++s) len[s] = static_cast<uint32_t>(s_len[s]);
  while (c < g1 * XP_LANES) {  // the same for all lanes of a half-wave
    const uint32_t w[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
    uint32_t bits = 0;
#pragma unroll
    for (int s = 0; s < 8; ++s) bits += (w[s] & 0xffffu) * len[s] + ((w[s] >> 16) & 0x0fffu) * len[s + 8];
    bits -= static_cast<uint32_t>(s_len[w[7] >> 28]);  // not the last symbol
    uint32_t words = (bits + XP_LIMIT - 1) / 32 + 1;
#pragma unroll
    for (int d = 16; d >= 1; d >>= 1) words += __shfl_xor(words, d, 32);
    if ((tid & 31) == 0) a.words[static_cast<int64_t>(row) * a.G + c / XP_LANES] = static_cast<int32_t>(words);
    c += kThreads;
    if (c < g1 * XP_LANES) {
      lo = *reinterpret_cast<const u32x4_any*>(counts + int64_t(c) * 8);
      hi = *reinterpret_cast<const u32x4_any*>(counts + int64_t(c) * 8 + 4);
    }
  }
}

// ---- the plan of a row by one workgroup: xp_encode_rows ----
__global__ void __launch_bounds__(kPlanThreads) encode_plan_kernel(EncodeArgs a) {
  __shared__ uint32_t s_hist[code::kSyms][kPlanThreads];  // per-thread counters
  __shared__ int32_t s_len[code::kSyms];
  __shared__ int32_t s_code[code::kSyms];
  __shared__ int32_t s_words[kMaxGroups + 1];          // words per group, then gstart
  __shared__ int64_t s_total;

  const int row = blockIdx.x;
  const int tid = threadIdx.x;
  const uint8_t* raw = a.raw + static_cast<int64_t>(row) * a.raw_stride;
  uint8_t* rec = a.rec + static_cast<int64_t>(row) * a.pitch;
  const int64_t n = a.n;
  const int chunk = a.chunk, G = a.G;

  // 1. Histogram of the exponent fields. Each thread counts into its own
  // LDS counters with atomic adds whose result is not returned: a plain
  // increment is a read and a write that the next increment of the same
  // counter must wait for, a chain of LDS round trips per byte.
  for (int s = 0; s < code::kSyms; ++s) s_hist[s][tid] = 0;
  constexpr int64_t kStep = int64_t(kPlanThreads) * 16;
  for (int64_t off0 = int64_t(tid) * 16; off0 < n; off0 += kStep * kPlanUnroll) {
    u32x4 v[kPlanUnroll];
#pragma unroll
    for (int u = 0; u < kPlanUnroll; ++u)
      if (off0 + u * kStep < n) v[u] = *reinterpret_cast<const u32x4*>(raw + off0 + u * kStep);
#pragma unroll
    for (int u = 0; u < kPlanUnroll; ++u) {
      if (off0 + u * kStep >= n) continue;
      const uint32_t w[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int b = 0; b < 4; ++b) atomicAdd(&s_hist[(w[k] >> (8 * b + 3)) & 15u][tid], 1u);
    }
  }
  __syncthreads();

  // 2. The code, and the LUT. Wave w sums symbol w's counters.
  static_assert(kPlanThreads / 64 == code::kSyms, "one wave per symbol");
  {
    const int sym = tid >> 6, part = tid & 63;
    uint32_t t = 0;
    for (int i = 0; i < kPlanThreads / 64; ++i) t += s_hist[sym][part * (kPlanThreads / 64) + i];
    for (int d = 32; d >= 1; d >>= 1) t += __shfl_xor(t, d, 64);
    if (part == 0) s_hist[sym][0] = t;
  }
  __syncthreads();
  if (tid < 64) {
    const int length = wave_code_lengths(s_hist[tid & 15][0]);
    const int code = wave_canonical_code(length);
    if (tid < code::kSyms) {
      s_len[tid] = length;
      s_code[tid] = code;
    }
  }
  __syncthreads();
  write_lut(s_len, s_code, a.lut + static_cast<int64_t>(row) * a.lut_stride, kPlanThreads);
  uint32_t lb[4];
  pack_lengths(s_len, lb);

  // 3. Words per group.
  const int per = chunk / 16;  // threads per chunk
  for (int g = tid; g < G; g += kPlanThreads) s_words[g] = 0;
  __syncthreads();
  // A chunk's pieces are all below n or all at or past it (n is a multiple
  // of the chunk), so each set of lanes shuffles together.
  for (int64_t off0 = int64_t(tid) * 16; off0 < n; off0 += kStep * kPlanUnroll) {
    u32x4 v[kPlanUnroll];
#pragma unroll
    for (int u = 0; u < kPlanUnroll; ++u)
      if (off0 + u * kStep < n) v[u] = *reinterpret_cast<const u32x4*>(raw + off0 + u * kStep);
#pragma unroll
    for (int u = 0; u < kPlanUnroll; ++u) {
      const int64_t off = off0 + u * kStep;
      if (off >= n) continue;
      add_chunk_words(v[u], off, chunk, per, lb, s_words, 0);
    }
  }
  __syncthreads();
  if (tid == 0) {  // exclusive scan into gstart
    int64_t t = 0;
    for (int g = 0; g < G; ++g) {
      const int32_t w = s_words[g];
      s_words[g] = static_cast<int32_t>(t);
      t += w;
    }
    s_words[G] = static_cast<int32_t>(t);
    s_total = t;
  }
  __syncthreads();
  const int64_t head = 4 * (int64_t(G) + 1) + n / 2;
  const int64_t nbytes = head + 4 * s_total;
  if (tid == 0) a.needed[row] = nbytes;
  if (nbytes > a.pitch) return;

  int32_t* gstart = reinterpret_cast<int32_t*>(rec);
  for (int g = tid; g <= G; g += kPlanThreads) gstart[g] = s_words[g];
  // Zero tail (nbytes and the pitch are multiples of 4).
  for (int64_t i = nbytes / 4 + tid; i < a.pitch / 4; i += kPlanThreads) reinterpret_cast<uint32_t*>(rec)[i] = 0;
}

// Waves that share a group's chunks, each a segment of all of them, where the
// groups are few. A chain of 512 symbols takes a wave 48 us however few
// groups there are; the state at a segment's start follows from the code
// lengths before it: a lane's bit position P is their sum, the words it has
// loaded number (P(last symbol) + LIMIT - 1) / 32 + 1, and a group's are the
// sum over its lanes. A word loaded early belongs to a symbol at most 8 before
// the start, so a wave walks those 8 without writing; the word that a start
// falls into is joined from both waves' bits in LDS (a segment has at least 64
// bits, so it ends in the next wave's).
// The sums and the 8 symbols are a quarter more work, so rows that fill the
// chip keep one wave for two whole groups. The whole call, without the check,
// for 1, 16, 32 and 64 rows of 128 groups: 67, 84, 106 and 161 us with one
// segment, 37, 66, 107 and 170 with four, 31, 61, 94 and 160 with eight (with
// the plan's second pass over the rows still in them).
constexpr int kSegments = 8;
constexpr int kMinSegment = 64;  // symbols: a block of loads
constexpr int64_t kSegmentGroups = 4096;

// SPLIT: the words per group come from encode_words_kernel; the workgroup
// sums those before its groups and writes its part of gstart and of the tail.
// SEG > 1: two groups per workgroup, cut into SEG segments.
template <bool SPLIT, int SEG>
__global__ void __launch_bounds__(SEG > 1 ? 64 * SEG : 256) encode_groups_kernel(EncodeArgs a, int blocks_per_row) {
  constexpr int kThreads = SEG > 1 ? 64 * SEG : xp::kThreads;
  constexpr int kGroupsPerBlock = SEG > 1 ? 2 : xp::kGroupsPerBlock;
  __shared__ uint32_t s_bits[SEG][64];  // SEG > 1: a lane's bits in each segment
  __shared__ uint32_t s_head[SEG][64];  // SEG > 1: the segment's bits of the word that its start falls into
  __shared__ int32_t s_len[code::kSyms];
  __shared__ uint32_t s_code[code::kSyms];  // code | length << 16
  __shared__ uint2 s_pair[code::kSyms * code::kSyms];  // see encode_pair
  __shared__ int32_t s_gstart[kGroupsPerBlock + 1];  // SPLIT: of the workgroup's groups, then the row's words
  __shared__ int32_t s_sum[2][kThreads / 64];

  const int row = blockIdx.x / blocks_per_row, part = blockIdx.x % blocks_per_row;
  const int tid = threadIdx.x;
  const uint8_t* raw = a.raw + static_cast<int64_t>(row) * a.raw_stride;
  uint8_t* rec = a.rec + static_cast<int64_t>(row) * a.pitch;
  const int64_t n = a.n;
  const int chunk = a.chunk, G = a.G;
  const int gfirst = part * kGroupsPerBlock;
  const int64_t head = 4 * (int64_t(G) + 1) + n / 2;
  if constexpr (SPLIT) {
    const int32_t* words = a.words + static_cast<int64_t>(row) * G;
    int32_t below = 0, all = 0;
    for (int g = tid; g < G; g += kThreads) {
      const int32_t w = words[g];
      all += w;
      below += g < gfirst ? w : 0;
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
      all += __shfl_xor(all, d, 64);
      below += __shfl_xor(below, d, 64);
    }
    if ((tid & 63) == 0) {
      s_sum[0][tid >> 6] = below;
      s_sum[1][tid >> 6] = all;
    }
    __syncthreads();
    below = all = 0;
#pragma unroll
    for (int w = 0; w < kThreads / 64; ++w) {
      below += s_sum[0][w];
      all += s_sum[1][w];
    }
    const int64_t nbytes = head + 4 * int64_t(all);
    if (tid == 0 && part == 0) a.needed[row] = nbytes;
    if (nbytes > a.pitch) return;  // the row does not fit: only its LUT and its size are written
    if (tid < kGroupsPerBlock) {
      for (int i = 0; i < tid; ++i) below += gfirst + i < G ? words[gfirst + i] : 0;
      s_gstart[tid] = below;
      if (gfirst + tid < G) reinterpret_cast<int32_t*>(rec)[gfirst + tid] = below;
    } else if (tid == kGroupsPerBlock) {
      s_gstart[tid] = all;
      if (part == 0) reinterpret_cast<int32_t*>(rec)[G] = all;
    }
    // Zero tail (nbytes and the pitch are multiples of 4), a stride per workgroup.
    for (int64_t i = nbytes / 4 + int64_t(part) * kThreads + tid; i < a.pitch / 4; i += int64_t(blocks_per_row) * kThreads)
      reinterpret_cast<uint32_t*>(rec)[i] = 0;
  } else {
    if (a.needed[row] > a.pitch) return;  // the row does not fit: the plan wrote nothing either
    const int32_t* gstart = reinterpret_cast<const int32_t*>(rec);
    if (tid < kGroupsPerBlock)
      s_gstart[tid] = gstart[gfirst + tid < G ? gfirst + tid : G];
    else if (tid == kGroupsPerBlock)
      s_gstart[tid] = gstart[G];
  }

  // 4. The code from the LUT (entry = symbol << 4 | length), then groups,
  // one per half-wave.
  const uint8_t* lut = a.lut + static_cast<int64_t>(row) * a.lut_stride;
  for (int x = tid; x < XP_LUT_BYTES; x += kThreads) {
    const uint32_t ent = lut[x];
    s_len[ent >> 4] = static_cast<int32_t>(ent & 15u);  // every entry of a symbol holds the same length
  }
  __syncthreads();
  if (tid < 64) {
    const int length = s_len[tid & 15];
    const int code = wave_canonical_code(length);
    if (tid < code::kSyms) s_code[tid] = static_cast<uint32_t>(code) | (static_cast<uint32_t>(length) << 16);
  }
  __syncthreads();
  static_assert(kThreads >= code::kSyms * code::kSyms, "a thread per pair of symbols");
  if (tid < code::kSyms * code::kSyms) {
    const uint32_t first = s_code[tid & 15], second = s_code[tid >> 4];
    const uint32_t l0 = first >> 16, l01 = l0 + (second >> 16);
    s_pair[tid] = make_uint2((first & 0xffffu) | ((second & 0xffffu) << l0), (l0 << 26) | l01);
  }
  __syncthreads();

  uint32_t* fixed = reinterpret_cast<uint32_t*>(rec + 4 * (int64_t(G) + 1));
  uint32_t* huff = reinterpret_cast<uint32_t*>(rec + head);
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const bool upper = lane >= 32;
  const uint32_t li = lane & 31;
  const uint32_t half_shift = upper ? 16u : 0u;
  const int mwords = chunk / 8;
  const uint32_t total = static_cast<uint32_t>(s_gstart[kGroupsPerBlock]);  // every word position is below it
  {
    const int pair_of_groups = SEG > 1 ? 0 : wave, seg = SEG > 1 ? wave : 0;
    const int g0 = gfirst + 2 * pair_of_groups;
    if (g0 >= G) return;  // SEG > 1: never
    const int g = g0 + (upper ? 1 : 0);
    const bool live = g < G;  // a spare half-wave walks the last group and writes nothing
    const int gg = live ? g : G - 1;
    const int length = chunk / SEG, begin = seg * length;  // of the wave's segment
    const uint8_t* src = raw + (int64_t(gg) * XP_LANES + li) * chunk + begin;
    uint32_t* fx = fixed + (int64_t(gg) * mwords + begin / 8) * XP_LANES + li;
    // Word positions within each half's group, both below 2^16 (a group's
    // words are at most 32 chunks of 9-bit codes), packed in one scalar
    // register: the lower half's in bits 0-15, the upper half's in 16-31
    // biased by kBias, so that lowering the upper half's count by the lower
    // half's refills of a symbol (at most 32) never borrows. A lane's word
    // positions are relative; gbase makes them absolute.
    constexpr uint32_t kBias = 64;
    const uint32_t gs_lo = static_cast<uint32_t>(s_gstart[2 * pair_of_groups]);
    const uint32_t gs_hi = static_cast<uint32_t>(s_gstart[2 * pair_of_groups + (g0 + 1 < G ? 1 : 0)]);
    const uint32_t gbase = upper ? gs_hi - kBias : gs_lo;
    uint32_t limit = live ? total : 0u;
    uint32_t offs = kBias << 16;
    // The decoder has fewer than LIMIT bits left before the symbol that starts
    // at bit P of the lane's stream exactly when the words it has loaded
    // number no more than (P + LIMIT - 1) / 32, so it loads one where that
    // quotient steps: where bit 5 of Q = P + LIMIT - 1 differs from the
    // symbol's before it (a symbol is shorter than 32 bits). Q mod 64 is kept
    // in bits 26-31, so that the step is a sign. The first symbol always
    // loads.
    uint32_t Q = uint32_t(XP_LIMIT - 1) << 26;  // of the next symbol
    uint32_t Qp = Q ^ 0x80000000u;              // of the symbol before (bits below 26 are not used)
    uint32_t acc = 0, accbits = 0;              // the bits of the word being filled
    uint32_t wcur = 0, wprev = 0;               // positions of the last word loaded and the one before
    bool head = false;                          // the next word complete is the one that the segment starts in
    // Two symbols at a time (`at` is 8 x (second * 16 + first)): a pair's
    // entry holds both codes in a row, their length l01 in bits 0-5 and the
    // first's in bits 26-31. Loads are at least three symbols apart (a load
    // leaves 32 bits or more, a symbol takes at most 9), so a pair has at
    // most one; and at most 18 bits, so it completes at most one word. That
    // word is the last one loaded, unless the next one has been loaded
    // already, as soon as 24 of its bits are there: unless the second symbol
    // starts before bit 24. Completing a word from a start of at most 23 takes
    // all 9 bits from exactly 23, where Q mod 32 = 31.
    // The loop is VALU bound: about 20 instructions a symbol, half of what
    // symbol by symbol with a two-entry queue of loaded words took. 256 rows
    // of 2 MiB: 485 -> 358 us (2.2 TB/s read and written); one row, a chain of
    // 512 symbols in 64 waves, 71 -> 48 us (in segments, see kSegments, 13). Reading a 16-byte piece's eight
    // entries ahead of its pairs changed neither.
    auto encode_pair = [&](uint32_t at) {
      const uint2 t = *reinterpret_cast<const uint2*>(reinterpret_cast<const uint8_t*>(s_pair) + at);
      const uint32_t q1 = Q + t.y;
      const bool r0 = static_cast<int32_t>(Q ^ Qp) < 0, r1 = static_cast<int32_t>(q1 ^ Q) < 0;
      auto place = [&](bool refill) {  // the word's rank among the refilling lanes of the half
        const unsigned long long mask = __builtin_amdgcn_ballot_w64(refill);
        const uint32_t m_lo = static_cast<uint32_t>(mask), m_hi = static_cast<uint32_t>(mask >> 32);
        const uint32_t n_lo = static_cast<uint32_t>(__popc(m_lo)), n_hi = static_cast<uint32_t>(__popc(m_hi));
        const uint32_t bases = offs - (n_lo << 16);
        offs += n_lo + (n_hi << 16);
        return __builtin_amdgcn_mbcnt_hi(
            m_hi, __builtin_amdgcn_mbcnt_lo(m_lo, __builtin_amdgcn_ubfe(bases, half_shift, 16u)));
      };
      const uint32_t p0 = place(r0), p1 = place(r1);
      wprev = r0 || r1 ? wcur : wprev;
      wcur = r0 ? p0 : wcur;
      wcur = r1 ? p1 : wcur;
      Q += t.y << 26;
      Qp = q1;
      const uint64_t shifted = static_cast<uint64_t>(t.x) << accbits;
      const uint32_t word = acc | static_cast<uint32_t>(shifted);
      const uint32_t bits = accbits + (t.y & 63u);
      const bool full = bits >= 32;
      if (full) {
        const bool alone = (q1 & 0x7C000000u) == 0x7C000000u;
        const uint32_t at_word = gbase + (alone ? wcur : wprev);
        if (SEG > 1 && head) {
          s_head[seg][lane] = word;
          head = false;
        } else if (at_word < limit) {
          huff[at_word] = word;
        }
      }
      acc = full ? static_cast<uint32_t>(shifted >> 32) : word;
      accbits = bits & 31u;
    };
    // A lane's values in blocks of 64 (four 16-byte loads back to back, so
    // each cache line of its chunk is fetched about twice instead of once
    // per 16 values), the next block loaded while this one is encoded.
    const int nv = SEG == 1 && chunk < 64 ? chunk / 16 : 4;  // loads per block
    u32x4 cur[4], nxt[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (j < nv) cur[j] = *reinterpret_cast<const u32x4*>(src + 16 * j);
    if constexpr (SEG > 1) {
      // The 16 values before the segment (the first segment: its own).
      const u32x4 pre = *reinterpret_cast<const u32x4*>(src - (seg > 0 ? 16 : 0));
      uint32_t lb[4];
      pack_lengths(s_len, lb);
      uint32_t bits = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        bits += sum_lengths4(cur[j].x, lb) + sum_lengths4(cur[j].y, lb) + sum_lengths4(cur[j].z, lb) +
                sum_lengths4(cur[j].w, lb);
      for (int i = 64; i < length; i += 16) {
        const u32x4 v = *reinterpret_cast<const u32x4*>(src + i);
        bits += sum_lengths4(v.x, lb) + sum_lengths4(v.y, lb) + sum_lengths4(v.z, lb) + sum_lengths4(v.w, lb);
      }
      s_bits[seg][lane] = bits;
      __syncthreads();
      uint32_t start = 0;
#pragma unroll
      for (int k = 0; k < SEG - 1; ++k) start += k < seg ? s_bits[k][lane] : 0u;
      if (seg > 0) {
        const uint32_t p8 = start - sum_lengths4(pre.z, lb) - sum_lengths4(pre.w, lb);  // of the 8th symbol before
        const uint32_t p9 = p8 - static_cast<uint32_t>(s_len[pre.y >> 27 & 15u]);
        Q = (p8 + XP_LIMIT - 1) << 26;
        Qp = (p9 + XP_LIMIT - 1) << 26;
        uint32_t loaded = (p9 + XP_LIMIT - 1) / 32 + 1;
#pragma unroll
        for (int d = 16; d >= 1; d >>= 1) loaded += __shfl_xor(loaded, d, 32);
        offs = static_cast<uint32_t>(__builtin_amdgcn_readlane(loaded, 0)) +
               ((static_cast<uint32_t>(__builtin_amdgcn_readlane(loaded, 32)) + kBias) << 16);
        accbits = p8 & 31u;
        const uint32_t to = limit;
        limit = 0;  // nothing is written
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const uint32_t ex = (k ? pre.w : pre.z) & 0x78787878u, z = ex | (ex >> 4);
          encode_pair(z & 0x7F8u);
          encode_pair((z >> 16) & 0x7F8u);
        }
        limit = to;
        acc = 0;
        head = accbits != 0;
      }
    }
    for (int i0 = 0; i0 < length; i0 += 16 * nv) {
      if (i0 + 16 * nv < length) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (j < nv) nxt[j] = *reinterpret_cast<const u32x4*>(src + i0 + 16 * nv + 16 * j);
      }
#pragma unroll
      for (int jv = 0; jv < 4; ++jv) {
        if (jv >= nv) break;
        const u32x4 v = cur[jv];
        const int i1 = i0 + 16 * jv;
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          // A byte's exponent field is bits 3-6: the pairs' table offsets are
          // bits 3-10 and 19-26 of the fields and the fields shifted down by 4.
          const uint32_t ex = w[k] & 0x78787878u, z = ex | (ex >> 4);
          encode_pair(z & 0x7F8u);
          encode_pair((z >> 16) & 0x7F8u);
          if (k & 1) {  // 8 values: one nibble word, value j in bits 4j..4j+3
            // Per byte, sign (bit 7) to bit 3 beside the mantissa (bits 0-2);
            // then two bytes' nibbles joined and the four pairs picked.
            const uint32_t x0 = w[k - 1], x1 = w[k];
            const uint32_t t0 = (x0 & 0x07070707u) | ((x0 >> 4) & 0x08080808u);
            const uint32_t t1 = (x1 & 0x07070707u) | ((x1 >> 4) & 0x08080808u);
            const uint32_t nib = __builtin_amdgcn_perm(t1 | (t1 >> 4), t0 | (t0 >> 4), 0x06040200u);
            if (live) fx[int64_t((i1 + 8 * (k >> 1)) / 8) * XP_LANES] = nib;
          }
        }
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) cur[j] = nxt[j];
    }
    // Words loaded and not complete: the one being filled if the last symbol
    // started at or after bit 1 - LIMIT = -8 of it, and the next one, all
    // zeros, if it started at or after bit 24.
    const int last = static_cast<int>(accbits) - static_cast<int>((Q - (Qp & 0xFC000000u)) >> 26);
    if constexpr (SEG > 1) {
      __syncthreads();
      if (seg < SEG - 1) {  // the next segment's start is in the word being filled, unless a word ends there
        const uint32_t at_word = gbase + (last >= 24 ? wprev : wcur);
        if (accbits != 0 && at_word < limit) huff[at_word] = acc | s_head[seg + 1][lane];
        return;
      }
    }
    if (last >= 24) {
      if (gbase + wprev < limit) huff[gbase + wprev] = acc;
      if (gbase + wcur < limit) huff[gbase + wcur] = 0;
    } else if (last >= -8) {
      if (gbase + wcur < limit) huff[gbase + wcur] = acc;
    }
  }
}

int64_t hist_parts(int64_t n) { return (n + kPartBytes - 1) / kPartBytes; }

}  // namespace
}  // namespace xp

using namespace xp;

extern "C" {

int64_t xp_encode_workspace_bytes(int64_t rows, int64_t n, int64_t chunk) {
  // Sizes that the encoder refuses need nothing, and must not overflow here.
  if (rows <= 0 || rows > INT32_MAX || chunk < 16 || chunk > 1024) return 0;
  const int64_t G = n / (chunk * XP_LANES);
  if (G < 1 || G > kMaxGroups) return 0;
  return 4 * rows * (hist_parts(n) * code::kSyms + G + (chunk >= kCountChunk ? n / chunk * 8 : 0));
}

int xp_encode_rows(const uint8_t* raw, int64_t rows, int64_t raw_stride, int64_t n, int64_t chunk, uint8_t* records,
                   int64_t pitch, uint8_t* luts, int64_t lut_stride, int64_t* needed, void* stream) {
  return xp_encode_rows_split(raw, rows, raw_stride, n, chunk, records, pitch, luts, lut_stride, needed, nullptr, 0,
                              stream);
}

int xp_encode_rows_split(const uint8_t* raw, int64_t rows, int64_t raw_stride, int64_t n, int64_t chunk,
                         uint8_t* records, int64_t pitch, uint8_t* luts, int64_t lut_stride, int64_t* needed,
                         void* work, int64_t work_bytes, void* stream) {
  XP_REQUIRE(rows >= 0 && rows <= INT32_MAX, "xp_encode_rows: rows=%lld", (long long)rows);
  if (rows == 0) return XP_OK;
  XP_REQUIRE(raw && records && luts && needed, "xp_encode_rows: null argument");
  XP_REQUIRE(chunk >= 16 && chunk <= 1024 && (chunk & (chunk - 1)) == 0,
             "xp_encode_rows: chunk=%lld (a power of two, 16..1024)", (long long)chunk);
  const int64_t group = chunk * XP_LANES;
  if (n <= 0 || n % group)
    return fail(XP_E_SHAPE, "row of %lld values is not a multiple of %lld", (long long)n, (long long)group);
  const int64_t G = n / group;
  XP_REQUIRE(G <= kMaxGroups, "xp_encode_rows: %lld groups per row (at most %d)", (long long)G, kMaxGroups);
  XP_REQUIRE(raw_stride >= n && raw_stride % 16 == 0 && aligned16(raw),
             "xp_encode_rows: raw rows must be 16-byte aligned with a stride of at least n");
  // A pitch below the header is a row that does not fit (needed > pitch), as
  // in xp_encode_row, not an argument error.
  XP_REQUIRE(pitch > 0 && pitch % 16 == 0 && aligned16(records),
             "xp_encode_rows: pitch %lld is not a positive multiple of 16", (long long)pitch);
  XP_REQUIRE(lut_stride >= XP_LUT_BYTES, "xp_encode_rows: lut_stride=%lld", (long long)lut_stride);
  EncodeArgs a{raw, raw_stride, n, static_cast<int>(chunk), static_cast<int>(G), records, pitch,
               luts, lut_stride, needed, nullptr, nullptr, 0, nullptr};
  const int64_t blocks = (G + kGroupsPerBlock - 1) / kGroupsPerBlock;
  XP_REQUIRE(rows * blocks <= INT32_MAX, "xp_encode_rows: %lld rows x %lld blocks", (long long)rows, (long long)blocks);
  const dim3 grid(static_cast<unsigned>(rows * blocks));
  if (!work) {
    hipLaunchKernelGGL(encode_plan_kernel, dim3(static_cast<unsigned>(rows)), dim3(kPlanThreads), 0,
                       as_stream(stream), a);
    if (int rc = check_launch("encode_plan_kernel")) return rc;
    hipLaunchKernelGGL((encode_groups_kernel<false, 1>), grid, dim3(kThreads), 0, as_stream(stream), a,
                       static_cast<int>(blocks));
    return check_launch("encode_groups_kernel");
  }
  const int64_t need = xp_encode_workspace_bytes(rows, n, chunk);
  XP_REQUIRE(work_bytes >= need && (reinterpret_cast<uintptr_t>(work) & 3) == 0,
             "xp_encode_rows_split: workspace of %lld B, needs %lld, 4-byte aligned", (long long)work_bytes,
             (long long)need);
  const int64_t parts = hist_parts(n);
  XP_REQUIRE(rows * parts <= INT32_MAX, "xp_encode_rows_split: %lld rows x %lld parts", (long long)rows,
             (long long)parts);
  a.parts = static_cast<int>(parts);
  a.hist = static_cast<uint32_t*>(work);
  a.words = static_cast<int32_t*>(work) + rows * parts * code::kSyms;
  a.counts = reinterpret_cast<uint32_t*>(a.words + rows * G);
  const bool counted = chunk >= kCountChunk;
  const dim3 plan_grid(static_cast<unsigned>(rows * parts));
  if (counted)
    hipLaunchKernelGGL(encode_count_kernel, plan_grid, dim3(kThreads), 0, as_stream(stream), a);
  else
    hipLaunchKernelGGL(encode_hist_kernel, plan_grid, dim3(kThreads), 0, as_stream(stream), a);
  if (int rc = check_launch(counted ? "encode_count_kernel" : "encode_hist_kernel")) return rc;
  // Counted chunks: a workgroup's threads take 8 groups at once.
  int64_t groups = counted ? kGroupsPerBlock : 1;
  while (groups < (counted ? kMaxGroups : kGroupsPerBlock) && rows * ((G + groups - 1) / groups) > kWordsBlocks)
    groups *= 2;
  const int64_t word_blocks = (G + groups - 1) / groups;
  XP_REQUIRE(rows * word_blocks <= INT32_MAX, "xp_encode_rows_split: %lld rows x %lld blocks", (long long)rows,
             (long long)word_blocks);
  const dim3 words_grid(static_cast<unsigned>(rows * word_blocks));
  if (counted)
    hipLaunchKernelGGL(encode_sizes_kernel, words_grid, dim3(kThreads), 0, as_stream(stream), a,
                       static_cast<int>(groups), static_cast<int>(word_blocks));
  else
    hipLaunchKernelGGL(encode_words_kernel, words_grid, dim3(kThreads), 0, as_stream(stream), a,
                       static_cast<int>(groups), static_cast<int>(word_blocks));
  if (int rc = check_launch(counted ? "encode_sizes_kernel" : "encode_words_kernel")) return rc;
  if (rows * G <= kSegmentGroups && chunk >= kSegments * kMinSegment) {
    const int64_t pairs = (G + 1) / 2;
    hipLaunchKernelGGL((encode_groups_kernel<true, kSegments>), dim3(static_cast<unsigned>(rows * pairs)),
                       dim3(64 * kSegments), 0, as_stream(stream), a, static_cast<int>(pairs));
  } else {
    hipLaunchKernelGGL((encode_groups_kernel<true, 1>), grid, dim3(kThreads), 0, as_stream(stream), a,
                       static_cast<int>(blocks));
  }
  return check_launch("encode_groups_kernel");
}

}  // extern "C"
