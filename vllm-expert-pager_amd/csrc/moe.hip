// Expert FFN on the slab for the prefill overflow path (and decode):
// fp8 e4m3 weights with 128x128 fp32 block scales, activations quantised to
// fp8 per token and 128-column group, MFMA fp8 grouped GEMMs, fused SiLU*up,
// and the single top-k combine.
//
// The reference hands expert_map to vLLM's fused fp8 MoE and intercepts its
// moe_sum so the top-k sum runs once over all chunks (experts.py:455-604).
// Here every (token, k) pair's expert output is computed independently of
// the other rows of its tile (an MFMA output element depends only on its own
// A row and B column), written once into a persistent buffer, and summed in
// k order in fp32 with one bf16 rounding at the end -- so a chunked run and
// a one-shot run give the same bits.
//
// Numerics of one pair follow the rounding sequence of a w8a8 block-fp8 MoE:
// x -> fp8 per 128-group (scale = max(amax, 1e-10) / 448, q = clamp(x / s));
// h = sum over K blocks of (xq . wq) * (sx * sw) in fp32; gate, up -> bf16;
// a = bf16(bf16(silu(gate)) * up) (silu is returned in bf16 and then
// multiplied, as vLLM's silu_and_mul does); a -> fp8 per 128-group; y
// likewise with w2;
// contribution = bf16(y * routed weight).
//
// Work decomposition: route lists the pairs of each slab slot in CSR form
// and cuts them into tiles of 64 pairs and wide tiles of 128 pairs of one
// slot. At prefill sizes gemm1 and gemm2 run one persistent workgroup per
// CU over (wide tile, column block) items (128 activation columns, 256
// output columns), so each column block of an expert's weights is read
// once, streamed through an LDS ring; for few pairs gemm1 takes 16 rows and 16
// columns of a tile, with the K blocks split over its waves (so a decode
// step of 8 pairs spreads over 256 workgroups), and gemm2 16 rows and 128
// output columns. Launch grids are sized from the shapes alone (bounds on
// the tile counts), so the sequence is graph-capturable; workgroups without
// live work exit at once.
#include <hip/hip_bf16.h>

#include <algorithm>
#include <mutex>
#include <type_traits>

#include "common.h"
#include "tile_split.h"

namespace xp {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr int kBM = 64;          // pairs per tile
constexpr int kWM = 2 * kBM;     // pairs per wide tile (the prefill GEMMs' work unit)
constexpr int kBN = 128;         // output columns per workgroup (one quant group for GEMM1)
constexpr int kKB = 128;         // K block = scale block = one MFMA K
constexpr int kThreads = 256;    // 4 waves, split along N (32 columns each)
constexpr int kRouteThreads = 1024;
constexpr int kMaxRouteSlots = 1024;
constexpr float kFp8Max = 448.0f;
constexpr float kEps = 1e-10f;

__device__ __forceinline__ float bf16_round(float v) { return __bfloat162float(__float2bfloat16(v)); }

__device__ __forceinline__ uint32_t bf16_bits(float v) {
  __hip_bfloat16 b = __float2bfloat16(v);
  return static_cast<uint32_t>(*reinterpret_cast<uint16_t*>(&b));
}

__device__ __forceinline__ float bf16_value(uint32_t u16) { return __uint_as_float(u16 << 16); }

__device__ __forceinline__ float quant_scale(float amax) { return fmaxf(amax, kEps) / kFp8Max; }

__device__ __forceinline__ float clamp_fp8(float v) { return fminf(fmaxf(v, -kFp8Max), kFp8Max); }

// Quantisation by one scale s: fp8(clamp(v / s)), e4m3 (OCP), to nearest even.
// The quotient is v * (1 / s) with one step of its remainder, three
// instructions where a division takes about ten and a quarter-rate one: v / s
// rounded correctly, as 1 / s is (Markstein 1990), where the remainder is
// exact. For a bf16 value and the scale of a bf16 maximum it is, except where
// both forms are below 2^-10, which rounds to zero of the same sign (all
// 32641 maxima with all values up to them, infinities among them, compared on
// the CPU). The remainder is taken as q * s - v, which keeps -0, and an
// infinite scale enters it as 0: finite values become 0, infinite ones NaN,
// as they do by division. Layers of 256 experts 2048 x 512: 1 token 14.0 -> 13.7
// us, 2048 tokens 254 -> 250, 8192 tokens 577 -> 566.
struct Quant {
  float inv, fin;
  __device__ __forceinline__ explicit Quant(float s) : inv(1.0f / s), fin(s < INFINITY ? s : 0.0f) {}
  __device__ __forceinline__ float operator()(float v) const {
    const float q = v * inv;
    return clamp_fp8(fmaf(-fmaf(q, fin, -v), inv, q));
  }
};

// Four quantised values as bytes, the first lowest.
__device__ __forceinline__ uint32_t fp8x4(float a, float b, float c, float d) {
  return static_cast<uint32_t>(
      __builtin_amdgcn_cvt_pk_fp8_f32(c, d, __builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false), true));
}

// Eight bf16 values (two per word) quantised.
__device__ __forceinline__ uint2 quant_words(const u32x4& raw, float s) {
  const Quant q(s);
  float v[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    v[2 * i] = q(bf16_value(raw[i] & 0xffffu));
    v[2 * i + 1] = q(bf16_value(raw[i] >> 16));
  }
  return make_uint2(fp8x4(v[0], v[1], v[2], v[3]), fp8x4(v[4], v[5], v[6], v[7]));
}

// a = bf16(bf16(act(g)) * u) for bf16 values g (gate) and u (up): the
// activation in fp32 as vLLM's activation kernels compute it, returned in
// the activation dtype (bf16), then the product of two bf16 values.
// SiLU: g / (1 + exp(-g)); GELU: g * 0.5 * (1 + erf(g / sqrt(2))).
template <int ACT>
__device__ __forceinline__ float act_and_mul(float g, float u) {
  static_assert(ACT == XP_ACT_SILU || ACT == XP_ACT_GELU, "activation");
  float a;
  if constexpr (ACT == XP_ACT_GELU)
    a = g * 0.5f * (1.0f + erff(g * 0.70710678118654752f));
  else
    a = g / (1.0f + expf(-g));
  return bf16_round(bf16_round(a) * u);
}

// The maximum of v over the 16 lanes of its DPP row (lanes 16r .. 16r + 15):
// quad swaps at lane distance 1 and 2, then the half-row and row mirrors,
// each a DPP operand of v_max, with no LDS round trip. Max is exact and
// order-free, so this equals a butterfly over lane distances 1, 2, 4 and 8.
// Every lane of the row must be active.
__device__ __forceinline__ float row16_max(float v) {
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, false)));   // quad [1,0,3,2]
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4E, 0xF, 0xF, false)));   // quad [2,3,0,1]
  v = fmaxf(v, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x141, 0xF, 0xF, false)));  // row_half_mirror
  return fmaxf(v, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x140, 0xF, 0xF, false)));  // row_mirror
}

// The maximum of v over the four lanes 16 apart (lane % 16 equal): each swap
// exchanges the odd rows (the upper half) of one copy with the even rows (the
// lower half) of the other, so the maximum of the two copies covers a pair.
__device__ __forceinline__ float quad16_max(float v) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// 16x16 output tile = A[16][128] . B[128][16] in fp8 e4m3. Lane l = 16q + j
// supplies 32 bytes of A row j and of B column j at K offset 32q; the
// instruction maps the bytes of A and B to K in the same way, so the dot
// products are those of the plain layout. Lane l receives C[4q + r][j].
// Zero scale operands select the unscaled instruction.
__device__ __forceinline__ f32x4 mfma_k128(const u32x4 (&a)[2], const u32x4 (&b)[2]) {
  const i32x8 av = {static_cast<int>(a[0].x), static_cast<int>(a[0].y), static_cast<int>(a[0].z),
                    static_cast<int>(a[0].w), static_cast<int>(a[1].x), static_cast<int>(a[1].y),
                    static_cast<int>(a[1].z), static_cast<int>(a[1].w)};
  const i32x8 bv = {static_cast<int>(b[0].x), static_cast<int>(b[0].y), static_cast<int>(b[0].z),
                    static_cast<int>(b[0].w), static_cast<int>(b[1].x), static_cast<int>(b[1].y),
                    static_cast<int>(b[1].z), static_cast<int>(b[1].w)};
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(av, bv, zero, 0, 0, 0, 0, 0, 0);
}

__device__ __forceinline__ void load32(const uint8_t* p, u32x4 (&v)[2]) {
  v[0] = *reinterpret_cast<const u32x4*>(p);
  v[1] = *reinterpret_cast<const u32x4*>(p + 16);
}

// ---- token quantisation: 256 threads per token, 16 lanes per group ----
__device__ __forceinline__ void quant_token(const uint16_t* __restrict__ x, int64_t H, uint8_t* __restrict__ xq,
                                            float* __restrict__ xs, int64_t t, int tid) {
  const uint16_t* row = x + t * H;
  for (int64_t c0 = tid * 8; c0 < H; c0 += 256 * 8) {
    const u32x4 raw = *reinterpret_cast<const u32x4*>(row + c0);
    float v[8];
    float amax = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[2 * i] = bf16_value(raw[i] & 0xffffu);
      v[2 * i + 1] = bf16_value(raw[i] >> 16);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) amax = fmaxf(amax, fabsf(v[i]));
    amax = row16_max(amax);
    const float s = quant_scale(amax);
    *reinterpret_cast<uint2*>(xq + t * H + c0) = quant_words(raw, s);
    if ((tid & 15) == 0) xs[t * (H / kKB) + c0 / kKB] = s;
  }
}

__global__ void __launch_bounds__(256) quant_tokens_kernel(const uint16_t* __restrict__ x, int64_t H,
                                                           uint8_t* __restrict__ xq, float* __restrict__ xs) {
  quant_token(x, H, xq, xs, blockIdx.x, threadIdx.x);
}

// Exclusive scan of three counters over a 1024-thread workgroup.
__device__ __forceinline__ int3 block_scan3(int3 v, int3* s_tot, int3* total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int3 in = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int ya = __shfl_up(in.x, off, 64), yb = __shfl_up(in.y, off, 64), yc = __shfl_up(in.z, off, 64);
    if (lane >= off) {
      in.x += ya;
      in.y += yb;
      in.z += yc;
    }
  }
  if (lane == 63) s_tot[wave] = in;
  __syncthreads();
  int3 base = make_int3(0, 0, 0), all = make_int3(0, 0, 0);
  for (int w = 0; w < kRouteThreads / 64; ++w) {
    const int3 t = s_tot[w];
    if (w < wave) {
      base.x += t.x;
      base.y += t.y;
      base.z += t.z;
    }
    all.x += t.x;
    all.y += t.y;
    all.z += t.z;
  }
  *total = all;
  return make_int3(base.x + in.x - v.x, base.y + in.y - v.y, base.z + in.z - v.z);
}

// ---- routing: CSR lists of the pairs of each slab slot, and the tiles ----
// offsets[slots + 1]; pairs[offsets[s] .. offsets[s+1]) = pair ids t*topk + k
// of slot s; tiles[0] = live tile count, then (slot, first pair position)
// per tile of kBM pairs; wide[0] = live wide-tile count, then (slot, first
// pair position, pair count) per wide tile of kWM pairs (wide may be null).
// Each wave counts a contiguous range of pairs into its own LDS histogram (no
// contention between waves), so a slot's list is ordered by wave range;
// dynamic LDS = 16 * slots ints.
constexpr int64_t kRouteOne = 4096;  // pairs up to which one workgroup routes
constexpr int kRouteBatch = kRouteOne / kRouteThreads;

// Slots of the pairs p0, p0 + STRIDE, ... (N of them; -1 for pairs at or past
// hi, unknown experts and experts without a slot; without a map, expert e
// has slot e). All id loads are issued before the first expert_map load, and
// all of those before any is used: two memory round trips in all rather than
// two per pair.
template <int N, int STRIDE>
__device__ __forceinline__ void route_slots(const void* ids, int eb, int64_t p0, int64_t hi,
                                            const int32_t* __restrict__ expert_map, int E, int slots, int (&sl)[N]) {
  int64_t e[N];
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const int64_t p = p0 + STRIDE * j;
    e[j] = p < hi ? load_id(ids, eb, p) : -1;
  }
#pragma unroll
  for (int j = 0; j < N; ++j)
    sl[j] = (e[j] >= 0 && e[j] < E) ? (expert_map ? expert_map[e[j]] : static_cast<int>(e[j])) : -1;
#pragma unroll
  for (int j = 0; j < N; ++j) sl[j] = sl[j] < slots ? sl[j] : -1;
}

__device__ __forceinline__ void route_block(const void* ids, int eb, int64_t npairs,
                                            const int32_t* __restrict__ expert_map, int E, int slots,
                                            int32_t* __restrict__ offsets, int32_t* __restrict__ pairs,
                                            int32_t* __restrict__ tiles, int32_t* __restrict__ wide, int* s_hist,
                                            int3* s_tot) {
  constexpr int kW = kRouteThreads / 64;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  for (int i = tid; i < kW * slots; i += kRouteThreads) s_hist[i] = 0;
  __syncthreads();
  const int64_t per = (npairs + kW - 1) / kW;
  const int64_t lo = wave * per, hi = lo + per < npairs ? lo + per : npairs;
  int* hist = s_hist + wave * slots;
  // A wave's range is at most one batch, kept in registers for the scatter.
  int sl[kRouteBatch];
  route_slots<kRouteBatch, 64>(ids, eb, lo + lane, hi, expert_map, E, slots, sl);
#pragma unroll
  for (int j = 0; j < kRouteBatch; ++j)
    if (sl[j] >= 0) atomicAdd(&hist[sl[j]], 1);
  __syncthreads();
  int c = 0;
  if (tid < slots) {
    for (int w = 0; w < kW; ++w) {  // per-wave counts -> per-wave starts within the slot
      const int v = s_hist[w * slots + tid];
      s_hist[w * slots + tid] = c;
      c += v;
    }
  }
  const int nt = (c + kBM - 1) / kBM, nw = (c + kWM - 1) / kWM;
  int3 total;
  const int3 off = block_scan3(make_int3(c, nt, nw), s_tot, &total);
  if (tid < slots) {
    offsets[tid] = off.x;
    for (int w = 0; w < kW; ++w) s_hist[w * slots + tid] += off.x;  // scatter cursors
    for (int i = 0; i < nt; ++i) {
      tiles[1 + 2 * (off.y + i)] = tid;
      tiles[2 + 2 * (off.y + i)] = off.x + i * kBM;
    }
    if (wide)
      for (int i = 0; i < nw; ++i) {
        wide[1 + 3 * (off.z + i)] = tid;
        wide[2 + 3 * (off.z + i)] = off.x + i * kWM;
        wide[3 + 3 * (off.z + i)] = c - i * kWM < kWM ? c - i * kWM : kWM;
      }
  }
  if (tid == 0) {
    offsets[slots] = total.x;
    tiles[0] = total.y;
    if (wide) wide[0] = total.z;
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kRouteBatch; ++j)
    if (sl[j] >= 0) pairs[atomicAdd(&hist[sl[j]], 1)] = static_cast<int32_t>(lo + lane + 64 * j);
}

__global__ void __launch_bounds__(kRouteThreads) route_kernel(const void* ids, int eb, int64_t npairs,
                                                              const int32_t* __restrict__ expert_map, int E,
                                                              int slots, int32_t* __restrict__ offsets,
                                                              int32_t* __restrict__ pairs,
                                                              int32_t* __restrict__ tiles,
                                                              int32_t* __restrict__ wide) {
  extern __shared__ int s_hist[];  // [16 waves][slots]
  __shared__ int3 s_tot[kRouteThreads / 64];
  route_block(ids, eb, npairs, expert_map, E, slots, offsets, pairs, tiles, wide, s_hist, s_tot);
}

// Quantisation and routing of one MoE call in one launch: workgroup 0
// routes, workgroup b >= 1 quantises tokens 4(b-1) .. 4(b-1)+3.
__global__ void __launch_bounds__(kRouteThreads) quant_route_kernel(const uint16_t* __restrict__ x, int64_t T,
                                                                    int64_t H, uint8_t* __restrict__ xq,
                                                                    float* __restrict__ xs, const void* ids, int eb,
                                                                    int64_t npairs,
                                                                    const int32_t* __restrict__ expert_map, int E,
                                                                    int slots, int32_t* __restrict__ offsets,
                                                                    int32_t* __restrict__ pairs,
                                                                    int32_t* __restrict__ tiles,
                                                                    int32_t* __restrict__ wide) {
  extern __shared__ int s_hist[];
  __shared__ int3 s_tot[kRouteThreads / 64];
  if (blockIdx.x == 0) {
    route_block(ids, eb, npairs, expert_map, E, slots, offsets, pairs, tiles, wide, s_hist, s_tot);
    return;
  }
  const int64_t t = (static_cast<int64_t>(blockIdx.x) - 1) * 4 + (threadIdx.x >> 8);
  if (t < T) quant_token(x, H, xq, xs, t, threadIdx.x & 255);
}

// ---- routing of many pairs: counted and scattered by several workgroups ----
//
// One workgroup is bound by its own LDS atomics and load round trips (two
// atomics a pair): 17 us at 16384 pairs over 256 slots, 81 us at 65536.
// Above kRouteOne pairs, `nb` workgroups each count a contiguous range of
// pairs into LDS and write their slot counts to the scratch after the wide
// list, beside the token quantisation where the call has one; a second
// launch of nb workgroups sums those counts (every workgroup for itself:
// nb x slots ints out of L2), scans them, and scatters its own range.
// 65536 pairs with 8192 tokens to quantise: 81 + 15 -> 19 + 9 us; 16384 with
// 2048: 17 + 5 -> 6 + 5 us. At 2664 pairs one workgroup takes 6 us beside the
// quantisation, as long as the two launches, so it keeps the small calls.
constexpr int64_t kRouteRange = 1024;   // pairs per workgroup, at least
constexpr int kRouteBlocks = 64;        // workgroups at most
constexpr int kCountBatch = 4;          // pairs a thread keeps in flight

// Workgroups that route npairs pairs (0: one workgroup, no count launch).
__host__ __device__ inline int route_blocks(int64_t npairs) {
  if (npairs <= kRouteOne) return 0;
  const int64_t nb = (npairs + kRouteRange - 1) / kRouteRange;
  return static_cast<int>(nb < kRouteBlocks ? nb : kRouteBlocks);
}

// Workgroups 0 .. nb - 1: hist[b][slots] = pairs of each slot in range b.
// The others quantise four tokens each (x null: none).
__global__ void __launch_bounds__(kRouteThreads) quant_count_kernel(const uint16_t* __restrict__ x, int64_t T,
                                                                    int64_t H, uint8_t* __restrict__ xq,
                                                                    float* __restrict__ xs, const void* ids, int eb,
                                                                    int64_t npairs, int nb,
                                                                    const int32_t* __restrict__ expert_map, int E,
                                                                    int slots, int32_t* __restrict__ hist) {
  __shared__ int s_count[kMaxRouteSlots];
  const int tid = threadIdx.x, b = blockIdx.x;
  if (b >= nb) {
    const int64_t t = (static_cast<int64_t>(b) - nb) * 4 + (tid >> 8);
    if (t < T) quant_token(x, H, xq, xs, t, tid & 255);
    return;
  }
  const int64_t per = (npairs + nb - 1) / nb;
  const int64_t lo = b * per, hi = lo + per < npairs ? lo + per : npairs;
  s_count[tid] = 0;
  __syncthreads();
  for (int64_t p = lo + tid; p < hi; p += kRouteThreads * kCountBatch) {
    int sl[kCountBatch];
    route_slots<kCountBatch, kRouteThreads>(ids, eb, p, hi, expert_map, E, slots, sl);
#pragma unroll
    for (int j = 0; j < kCountBatch; ++j)
      if (sl[j] >= 0) atomicAdd(&s_count[sl[j]], 1);
  }
  __syncthreads();
  if (tid < slots) hist[static_cast<int64_t>(b) * slots + tid] = s_count[tid];
}

// route_kernel's results from the counts, by nb = gridDim.x workgroups;
// workgroup 0 writes offsets and tiles, the last one the wide tiles.
__global__ void __launch_bounds__(kRouteThreads) route_scatter_kernel(
    const void* ids, int eb, int64_t npairs, const int32_t* __restrict__ expert_map, int E, int slots,
    const int32_t* __restrict__ hist, int32_t* __restrict__ offsets, int32_t* __restrict__ pairs,
    int32_t* __restrict__ tiles, int32_t* __restrict__ wide) {
  __shared__ int s_cur[kMaxRouteSlots];
  __shared__ int3 s_tot[kRouteThreads / 64];
  const int tid = threadIdx.x, b = blockIdx.x, nb = gridDim.x;
  const int64_t per = (npairs + nb - 1) / nb;
  const int64_t lo = b * per, hi = lo + per < npairs ? lo + per : npairs;
  int first[kCountBatch];  // the first pairs' slots, requested before the counts
  route_slots<kCountBatch, kRouteThreads>(ids, eb, lo + tid, hi, expert_map, E, slots, first);
  int c = 0, before = 0;
  if (tid < slots) {
#pragma unroll 8
    for (int i = 0; i < nb; ++i) {
      const int v = hist[static_cast<int64_t>(i) * slots + tid];
      c += v;
      before += i < b ? v : 0;
    }
  }
  const int nt = (c + kBM - 1) / kBM, nw = (c + kWM - 1) / kWM;
  int3 total;
  const int3 off = block_scan3(make_int3(c, nt, nw), s_tot, &total);
  if (tid < slots) {
    s_cur[tid] = off.x + before;
    if (b == 0) {
      offsets[tid] = off.x;
      for (int i = 0; i < nt; ++i) {
        tiles[1 + 2 * (off.y + i)] = tid;
        tiles[2 + 2 * (off.y + i)] = off.x + i * kBM;
      }
    }
    if (b == nb - 1)
      for (int i = 0; i < nw; ++i) {
        wide[1 + 3 * (off.z + i)] = tid;
        wide[2 + 3 * (off.z + i)] = off.x + i * kWM;
        wide[3 + 3 * (off.z + i)] = c - i * kWM < kWM ? c - i * kWM : kWM;
      }
  }
  if (tid == 0 && b == 0) {
    offsets[slots] = total.x;
    tiles[0] = total.y;
  }
  if (tid == 0 && b == nb - 1) wide[0] = total.z;
  __syncthreads();
  for (int64_t p = lo + tid; p < hi; p += kRouteThreads * kCountBatch) {
    int sl[kCountBatch];
    if (p == lo + tid) {
#pragma unroll
      for (int j = 0; j < kCountBatch; ++j) sl[j] = first[j];
    } else {
      route_slots<kCountBatch, kRouteThreads>(ids, eb, p, hi, expert_map, E, slots, sl);
    }
#pragma unroll
    for (int j = 0; j < kCountBatch; ++j)
      if (sl[j] >= 0) pairs[atomicAdd(&s_cur[sl[j]], 1)] = static_cast<int32_t>(p + kRouteThreads * j);
  }
}

struct Tile {
  int slot, first, count;
};

// Work item of a 1-D GEMM grid of ncols column blocks per tile, laid out so
// that every column block of a tile runs on the same XCD (workgroup L is
// dispatched to XCD L % 8): the tile's token rows and its expert's weight
// rows are then read into one L2. Tiles t, t + 8, ... belong to XCD t % 8.
__device__ __forceinline__ void xcd_item(int ncols, int& tile, int& col) {
  const int L = blockIdx.x, xcd = L & 7, j = L >> 3;
  tile = (j / ncols) * 8 + xcd;
  col = j - (j / ncols) * ncols;
}

__device__ __forceinline__ bool load_tile_at(int i, const int32_t* tiles, const int32_t* offsets, Tile& t) {
  if (i >= tiles[0]) return false;
  t.slot = tiles[1 + 2 * i];
  t.first = tiles[2 + 2 * i];
  const int end = offsets[t.slot + 1];
  t.count = end - t.first < kBM ? end - t.first : kBM;
  return true;
}

// Prefill-sized calls multiply wide tiles (up to kWM pairs of one slot), so
// that each column block of an expert's weights is read by one workgroup.
// route writes their list after the tile list (wide_list_offset).

// Bounds on the tile and wide-tile counts of npairs pairs over `slots`
// slots (each slot's last tile may be partial).
__host__ __device__ inline int64_t tile_bound(int64_t npairs, int64_t slots) {
  if (npairs <= 0 || slots <= 0) return 0;
  return (npairs + kBM - 1) / kBM + (slots < npairs ? slots : npairs);
}
__host__ __device__ inline int64_t wide_bound(int64_t npairs, int64_t slots) {
  if (npairs <= 0 || slots <= 0) return 0;
  return (npairs + kWM - 1) / kWM + (slots < npairs ? slots : npairs);
}

// The wide-tile list inside the tiles buffer, after the tile list's
// 1 + 2 * tile_bound ints: [0] = count, then (slot, first pair position,
// pair count) per wide tile.
__host__ __device__ inline int64_t wide_list_offset(int64_t npairs, int64_t slots) {
  return 1 + 2 * tile_bound(npairs, slots);
}

// The counts of the routing workgroups, after the wide list's 1 + 3 *
// wide_bound ints: [workgroup][slot].
__host__ __device__ inline int64_t route_hist_offset(int64_t npairs, int64_t slots) {
  return wide_list_offset(npairs, slots) + 1 + 3 * wide_bound(npairs, slots);
}

// Workspace of xp_moe_experts: bf16 activations, their per-16-column
// maxima, the fp8 activations and their per-128-column scales.
struct Work {
  uint16_t* a16;   // [npairs][I]
  float* amax16;   // [npairs][I/16]
  uint8_t* act;    // [npairs][I]
  float* acts;     // [npairs][I/128]
};

inline int64_t align256(int64_t n) { return (n + 255) & ~int64_t(255); }

inline int64_t work_layout(int64_t npairs, int64_t I, Work* w, uint8_t* base) {
  const int64_t sz[4] = {align256(npairs * I * 2), align256(npairs * (I / 16) * 4), align256(npairs * I),
                         align256(npairs * (I / kKB) * 4)};
  if (w) {
    w->a16 = reinterpret_cast<uint16_t*>(base);
    w->amax16 = reinterpret_cast<float*>(base + sz[0]);
    w->act = base + sz[0] + sz[1];
    w->acts = reinterpret_cast<float*>(base + sz[0] + sz[1] + sz[2]);
  }
  return sz[0] + sz[1] + sz[2] + sz[3];
}

constexpr int kWideTiles = 64;  // tile bound from which gemm1 uses the wide workgroups
constexpr int kNarrowChunk = 4; // K blocks per load chunk of the small-batch GEMMs
constexpr int kMaxKB = 64;    // K blocks a workgroup keeps row scales for (H, I <= 8192)

// ---- prefill GEMMs: persistent workgroups over wide tiles ----
//
// A work item is (wide tile, column block). Every XCD takes its share of the
// wide-tile list (tile_split.h), a tile's column blocks consecutive; workgroup
// b runs on XCD b % 8 and takes that XCD's items l, l + nl, l + 2 nl, ... (l =
// b / 8, nl = gridDim.x / 8), so a tile's column blocks run side by side on one
// XCD and its token rows are read into one L2, and the tiles of an expert with
// more than kWM pairs read its weight rows into one L2 at about the same time.
//
// The weight rows are the MFMA's A operand and the token rows its B operand,
// so a lane's four outputs are four columns of one token row: one scale read
// and one scale product per subtile and K block instead of four, and packed
// words instead of single values into the epilogues' LDS stages. Every
// output is the same sum of the same products either way. Both changes
// together, 2048 x 512 experts of 256 at top-8, skewed routing: 8192 tokens
// gemm1 413 -> 356 us and gemm2 221 -> 203 us, 2048 tokens 176 -> 169 and
// 86 -> 83 us.
//
// The operands stream through a ring of kRing LDS stages that global-to-LDS
// loads fill without passing through registers: a stage holds one K block
// of the item's weight rows, of the tile's A rows and of the A rows' scales.
// Each wave keeps the loads of the next kRing - 1 blocks in flight while it
// multiplies one, and the stream runs on across items: the next item's rows
// are looked up during the current item's first steps and its first blocks
// are requested during the last, so the epilogue and the next item's set-up
// overlap the loads.
//
// Vector memory operations complete in issue order, so "block k has landed"
// is "at most the loads this wave issued in the last step are in flight"
// (s_waitcnt vmcnt; the count depends on the item, see issue()).
// That holds only if nothing is issued after a step's operand loads, and if
// the compiler adds no waits of its own: every other load in the loop goes
// to LDS or through the scalar cache, and the epilogue's global stores are
// issued at the start of the next item's first step.
constexpr int kRing = 3;
constexpr int kAhead = kRing - 1;  // blocks requested ahead of the one multiplied
constexpr int kRowB = kKB;         // bytes of one operand row's K block (fp8)
constexpr int kGemmWaves = 8;      // waves of a prefill GEMM workgroup
constexpr int kMinSteps = 4;       // steps per item at least (the next item's set-up takes 3)

// This wave's loads but the last N have landed and its LDS writes are done;
// then the workgroup meets. A plain s_barrier: the fence of __syncthreads
// would also wait for the loads in flight.
template <int N>
__device__ __forceinline__ void ring_barrier() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// ring_barrier<n> for a wave-uniform n in [lo, hi]: the loads a wave issues
// per step depend on the item (see the prefill GEMMs), so the count left in
// flight is chosen at run time from the immediates the wait takes.
template <int LO, int HI>
__device__ __forceinline__ void ring_barrier_n(int n) {
  if constexpr (LO >= HI) {
    ring_barrier<HI>();
  } else {
    if (n <= LO)
      ring_barrier<LO>();
    else
      ring_barrier_n<LO + 1, HI>(n);
  }
}

__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const void*)p));
}
// A wave-uniform 64-bit address in scalar registers. The readfirstlane
// builtin returns int: each half is taken as uint32_t before widening, or a
// low half with bit 31 set would sign-extend into the high half.
__device__ __forceinline__ uint64_t uniform_ptr(const void* p) {
  const uint64_t v = reinterpret_cast<uint64_t>(p);
  const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v)));
  const uint32_t hi = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v >> 32)));
  return static_cast<uint64_t>(lo) | (static_cast<uint64_t>(hi) << 32);
}
// One piece per lane from global memory into LDS: lane l's 16 (4) bytes, at
// base + off (scalar base, 32-bit vector offset), land at dst + 16 l (4 l);
// base and dst are the same for the whole wave. Written in assembly so that
// the compiler does not track these loads: it would make every LDS access
// wait for all of them. M0 (the LDS destination) is restored afterwards.
__device__ __forceinline__ void dma16(const void* base, uint32_t off, void* dst) {
  uint32_t saved;
  asm volatile(
      "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0"
      : "=&s"(saved)
      : "v"(off), "s"(uniform_ptr(base)), "s"(__builtin_amdgcn_readfirstlane(lds_addr(dst)))
      : "memory");
}
// dma16 marked non-temporal, for weight rows that are read once per launch:
// they should not push the activation rows (re-read by every column block of a
// tile) out of the caches. Where experts have several tiles, each reads the
// rows again, and marked rows are no longer in its L2: dma_weights<false>.
// Whole layers of 256 experts 2048 x 512 at top-8, marked and not, by the mean
// pairs per expert: 16 (512 tokens) 177 and 186 us, 64 251 and 248, 128 372 and
// 346, 256 566 and 533. Through chunks of 64 of these experts 16 (512 tokens)
// 245 and 255, 32 295 and 305, 64 406 and 403, 128 474 and 463; of 16 experts
// 16 639 and 652, 32 793 and 803, 64 882 and 883. 23 tokens (4 layers) 287 and
// 305, 333 tokens of 64 experts 97 and 101. So the line is a mean of one whole
// tile per expert (stream_weights): of the experts that the pairs spread over,
// not of the slots of the slab, which holds a chunk of them. Chosen per item,
// by a branch around the loads, it cost the small calls 20%.
__device__ __forceinline__ void dma16_stream(const void* base, uint32_t off, void* dst) {
  uint32_t saved;
  asm volatile(
      "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt\n\ts_mov_b32 m0, %0"
      : "=&s"(saved)
      : "v"(off), "s"(uniform_ptr(base)), "s"(__builtin_amdgcn_readfirstlane(lds_addr(dst)))
      : "memory");
}
template <bool STREAM>
__device__ __forceinline__ void dma_weights(const void* base, uint32_t off, void* dst) {
  if constexpr (STREAM)
    dma16_stream(base, off, dst);
  else
    dma16(base, off, dst);
}
inline bool stream_weights(int64_t npairs, int64_t num_experts) { return npairs < num_experts * kWM; }
__device__ __forceinline__ void dma4(const void* base, uint32_t off, void* dst) {
  uint32_t saved;
  asm volatile(
      "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2\n\ts_mov_b32 m0, %0"
      : "=&s"(saved)
      : "v"(off), "s"(uniform_ptr(base)), "s"(__builtin_amdgcn_readfirstlane(lds_addr(dst)))
      : "memory");
}

// Stage rows are 128 bytes; 16-byte piece p of row r sits at slot p ^ (r & 7),
// so the 8 lanes that read one piece of 8 consecutive rows use distinct
// banks. A load of 8 rows writes slot l & 7 of row l / 8 from lane l, which
// therefore fetches global piece (l & 7) ^ (row & 7).
__device__ __forceinline__ int swizzled_piece(int lane) { return (lane & 7) ^ ((lane >> 3) & 7); }

// A lane's MFMA operand: bytes 32q .. 32q + 31 of stage row `row`.
__device__ __forceinline__ void read_frag(const uint8_t* stage, int row, int q, u32x4 (&v)[2]) {
  const uint8_t* r = stage + row * kRowB;
  const int s = row & 7;
  v[0] = *reinterpret_cast<const u32x4*>(r + (((2 * q) ^ s) << 4));
  v[1] = *reinterpret_cast<const u32x4*>(r + (((2 * q + 1) ^ s) << 4));
}

template <int N>
using Int = std::integral_constant<int, N>;

// Calls f(Int<n>{}) for the tile's subtile count n in 1..kWM/16: the K loop
// is compiled once per count, without branches and with no more
// accumulators than it needs.
template <int N, typename F>
__device__ __forceinline__ void with_subtiles_from(int nmi, F&& f) {
  if constexpr (N >= kWM / 16) {
    f(Int<kWM / 16>{});
  } else {
    if (nmi <= N)
      f(Int<N>{});
    else
      with_subtiles_from<N + 1>(nmi, f);
  }
}

template <typename F>
__device__ __forceinline__ void with_subtiles(int nmi, F&& f) {
  with_subtiles_from<1>(nmi, f);
}

struct Item {
  int slot, first, count, col;  // count 0: no item
};

// Candidate n of this workgroup: item j = l + n * nl of its XCD, i.e. the
// XCD's wide tile j / ncols (see tile_split.h) and column block j % ncols. Its
// list entry is read through the scalar cache (the list does not change
// during the call).
template <bool HALVES>
__device__ __forceinline__ Item item_fetch(int n, int ncols, const int32_t* __restrict__ wide, int64_t wmax) {
  const int jj = (static_cast<int>(blockIdx.x) >> 3) + n * (static_cast<int>(gridDim.x) >> 3);
  const int live = wide[0] < wmax ? wide[0] : static_cast<int>(wmax);
  const int t = jj / ncols;
  const int w = __builtin_amdgcn_readfirstlane(xcd_tile(live, static_cast<int>(blockIdx.x) & 7, t, HALVES));
  Item it;
  it.col = __builtin_amdgcn_readfirstlane(jj - t * ncols);
  it.slot = it.first = it.count = 0;
  if (w < live) {
    it.slot = wide[1 + 3 * static_cast<int64_t>(w)];
    it.first = wide[2 + 3 * static_cast<int64_t>(w)];
    it.count = wide[3 + 3 * static_cast<int64_t>(w)];
  }
  return it;
}

// The pairs of an item's rows (padding rows repeat its first pair) into
// s_pn, by waves 0 and 1.
__device__ __forceinline__ void request_pairs(const Item& it, const int32_t* __restrict__ pairs, int* s_pn) {
  const int tid = threadIdx.x, wave = tid >> 6;
  if (wave < kWM / 64) dma4(pairs + it.first, 4 * (tid < it.count ? tid : 0), s_pn + 64 * wave);
}

// s_pair (pair or -1 past the count) and s_row (the operand row, pair / div)
// from s_pn. Pairs are clamped to [0, npairs) before they address anything.
__device__ __forceinline__ void put_rows(const Item& it, const int* s_pn, int div, int64_t npairs, int* s_pair,
                                         int* s_row) {
  const int tid = threadIdx.x;
  if (tid < kWM) {
    const int p = s_pn[tid];
    const int c = p < 0 ? 0 : (p >= npairs ? static_cast<int>(npairs - 1) : p);
    s_pair[tid] = tid < it.count && c == p ? p : -1;
    s_row[tid] = c / div;
  }
}

// Per-lane byte offsets of a wave's A-row and A-scale loads for an item with
// operand rows s_row (A rows of lda bytes, KB scales per row): A stage rows
// 16 wave + 8 i + lane / 8 (i = 0, 1), scale rows 64 (wave & 1) + lane.
struct AOffsets {
  uint32_t a[2];
  uint32_t s;
};

__device__ __forceinline__ AOffsets a_offsets(const int* s_row, int64_t lda, int KB) {
  const int wave = static_cast<int>(threadIdx.x) >> 6, lane = static_cast<int>(threadIdx.x) & 63;
  AOffsets o;
#pragma unroll
  for (int i = 0; i < 2; ++i)
    o.a[i] = static_cast<uint32_t>(s_row[16 * wave + 8 * i + (lane >> 3)] * lda + 16 * swizzled_piece(lane));
  o.s = static_cast<uint32_t>(s_row[64 * (wave & 1) + lane] * KB * 4);
  return o;
}

// GEMM1 at prefill sizes: gate and up for 128 activation columns of a wide
// tile per item; each wave owns 16 columns (16 gate and 16 up rows) and runs
// the K blocks in order, so a column's value does not depend on the
// workgroup width or the tile height. Then a = bf16(bf16(silu(bf16 gate)) *
// bf16 up) is quantised to fp8 per row over the workgroup's 128 columns, one
// scale group. Only the 16-row subtiles that hold pairs are multiplied.
template <int ACT, bool STREAM>
__global__ void __launch_bounds__(kGemmWaves * 64) gemm1_kernel(const uint8_t* __restrict__ xq,
                                                               const float* __restrict__ xs, int64_t H, int64_t I,
                                                               int topk, const uint8_t* __restrict__ w13,
                                                               const float* __restrict__ w13_scale,
                                                               const int32_t* __restrict__ pairs,
                                                               const int32_t* __restrict__ wide, int64_t wmax,
                                                               int64_t npairs, Work work) {
  constexpr int NW = kGemmWaves, NT = NW * 64, NC = NW * 16;
  constexpr int NB = 2 * NC;       // weight rows per item: per wave 16 gate, then 16 up
  static_assert(NC == kKB, "a workgroup covers one 128-column scale group of the activations");
  __shared__ __attribute__((aligned(16))) uint8_t s_b[kRing][NB * kRowB];
  __shared__ __attribute__((aligned(16))) uint8_t s_a[kRing][kWM * kRowB];
  __shared__ __attribute__((aligned(16))) float s_s[kRing][kWM];
  __shared__ int s_pn[kWM];
  __shared__ int s_row[2][kWM];
  __shared__ int s_pair[2][kWM];
  __shared__ float s_sw[2][2 * kMaxKB];  // gate (first KB) and up weight scales per K block, two items
  __shared__ float s_m[NW][kWM];         // row maxima per wave (16 columns)
  __shared__ float s_q[kWM];             // row scales of the activations

  const int ncols = static_cast<int>(I / NC);
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int q = lane >> 4, j = lane & 15;
  const int KB = static_cast<int>(H / kKB), KS = KB > kMinSteps ? KB : kMinSteps;

  Item cur = item_fetch<STREAM>(0, ncols, wide, wmax);
  if (cur.count == 0) return;
  Item nxt = item_fetch<STREAM>(1, ncols, wide, wmax);
  int n = 2;

  // Weight-row loads: load i of a wave covers its stage rows 8i .. 8i + 7,
  // gate rows for i < 2 and up rows (I rows further) for i >= 2.
  uint32_t boff[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    boff[i] = static_cast<uint32_t>(((i >= 2 ? I : 0) + 16 * wave + 8 * (i & 1) + (lane >> 3)) * H +
                                    16 * swizzled_piece(lane));
  auto wbase = [&](const Item& it) {
    return w13 + (static_cast<int64_t>(it.slot) * 2 * I + static_cast<int64_t>(it.col) * NC) * H;
  };
  // Weight scales of an item into s_sw (waves 0 and 1): the workgroup's gate
  // and up rows each lie in one 128-row scale block.
  auto request_weight_scales = [&](const Item& it, float* dst) {
    if (wave < 2) {
      const int i = tid < 2 * KB ? tid : 2 * KB - 1;
      const int64_t blk = static_cast<int64_t>(it.slot) * (2 * I / kKB) + (i < KB ? 0 : I / kKB) + it.col;
      dma4(w13_scale, static_cast<uint32_t>(4 * (blk * KB + (i < KB ? i : i - KB))), dst + 64 * wave);
    }
  };
  // Block kb of an item with nmi live subtiles into `stage`: every wave its
  // 32 weight rows; wave w its A rows 16w .. 16w + 15 only when they hold
  // pairs (w < nmi); waves 0 and 1 the A rows' scales (wave 1's half only
  // when rows 64 and up hold pairs). Returns the loads this wave issued,
  // which the wait before the block after next leaves in flight.
  auto issue = [&](int stage, const uint8_t* wb, const AOffsets& ao, int kb, int nmi) {
    const uint8_t* bsrc = wb + kb * kRowB;
#pragma unroll
    for (int i = 0; i < 4; ++i) dma_weights<STREAM>(bsrc, boff[i], s_b[stage] + (32 * wave + 8 * i) * kRowB);
    int ops = 4;
    if (wave < nmi) {
      const uint8_t* asrc = xq + kb * kRowB;
#pragma unroll
      for (int i = 0; i < 2; ++i) dma16(asrc, ao.a[i], s_a[stage] + (16 * wave + 8 * i) * kRowB);
      ops += 2;
    }
    if (wave == 0 || (wave == 1 && nmi > 4)) {
      dma4(xs + kb, ao.s, &s_s[stage][64 * wave]);
      ops += 1;
    }
    return ops;
  };
  // The fp8 rows and scales of the previous item, staged in LDS.
  int out_cb = 0, out_c0 = 0, out_rows = 0;
  auto copy_out = [&](const uint8_t* stg) {
    if (tid < out_rows) {
      const int p = s_pair[out_cb][tid];
      if (p >= 0) work.acts[static_cast<int64_t>(p) * (I / kKB) + out_c0 / kKB] = s_q[tid];
    }
    // 16 bytes per thread and pass: 8 threads per row.
    for (int i = tid; i < out_rows * (kKB / 16); i += NT) {
      const int row = i >> 3, piece = i & 7;
      const int p = s_pair[out_cb][row];
      if (p >= 0)
        *reinterpret_cast<u32x4*>(work.act + static_cast<int64_t>(p) * I + out_c0 + piece * 16) =
            *reinterpret_cast<const u32x4*>(stg + row * kRowB + ((piece ^ (row & 7)) << 4));
    }
  };

  request_pairs(cur, pairs, s_pn);
  request_weight_scales(cur, s_sw[0]);
  ring_barrier<0>();
  put_rows(cur, s_pn, topk, npairs, s_pair[0], s_row[0]);
  lds_barrier();
  AOffsets ao_cur = a_offsets(s_row[0], H, KB), ao_nxt = ao_cur;
  issue(0, wbase(cur), ao_cur, 0, (cur.count + 15) >> 4);
  int last_ops = issue(1, wbase(cur), ao_cur, KB > 1 ? 1 : 0, (cur.count + 15) >> 4);

  int st = 0;  // stage of the current step
  int cb = 0;  // row set of the current item
  for (;;) {
    const int nb = cb ^ 1;
    const bool more = nxt.count > 0;
    const uint8_t* wb_cur = wbase(cur);
    const uint8_t* wb_nxt = more ? wbase(nxt) : wb_cur;
    const int nmi = (cur.count + 15) >> 4, nmi_nxt = (nxt.count + 15) >> 4;
    Item after = nxt;

    with_subtiles(nmi, [&](auto nmi_c) {
      constexpr int MI = decltype(nmi_c)::value;
      f32x4 acc[MI][2];
#pragma unroll
      for (int mi = 0; mi < MI; ++mi) acc[mi][0] = acc[mi][1] = f32x4{0.f, 0.f, 0.f, 0.f};

      for (int k = 0; k < KS; ++k) {
        ring_barrier_n<4, 7>(last_ops);  // block k is in stage st
        const int sn = st == 0 ? kRing - 1 : st - 1;  // the stage multiplied one step ago
        if (k == 0 && out_rows > 0) {
          copy_out(s_a[sn]);  // staged there by the previous item's epilogue
          out_rows = 0;
          lds_barrier();
        }
        // The next item: its pairs and the entry of the one after (step 0),
        // its rows (1), its A offsets and weight scales (2).
        if (more) {
          if (k == 0) {
            request_pairs(nxt, pairs, s_pn);
            after = item_fetch<STREAM>(n, ncols, wide, wmax);
          } else if (k == 1) {
            put_rows(nxt, s_pn, topk, npairs, s_pair[nb], s_row[nb]);
          } else if (k == 2) {
            ao_nxt = a_offsets(s_row[nb], H, KB);
            request_weight_scales(nxt, s_sw[nb]);
          }
        }
        // Block k + kAhead of this item, or the next item's first blocks.
        const int blk = k + kAhead;
        if (blk < KS || !more)
          last_ops = issue(sn, wb_cur, ao_cur, blk < KB ? blk : KB - 1, nmi);
        else
          last_ops = issue(sn, wb_nxt, ao_nxt, blk - KS < KB ? blk - KS : KB - 1, nmi_nxt);
        if (k < KB) {
          const float g = s_sw[cb][k], u = s_sw[cb][KB + k];
          u32x4 bg[2], bu[2];
          read_frag(s_b[st], 32 * wave + j, q, bg);
          read_frag(s_b[st], 32 * wave + 16 + j, q, bu);
          // Subtile mi + 1's A rows and scales are read while subtile mi
          // multiplies.
          u32x4 a[2][2];
          float sa[2];
          auto fetch = [&](int mi, int slot) {
            read_frag(s_a[st], 16 * mi + j, q, a[slot]);
            sa[slot] = s_s[st][16 * mi + j];
          };
          fetch(0, 0);
#pragma unroll
          for (int mi = 0; mi < MI; ++mi) {
            const int c = mi & 1;
            if (mi + 1 < MI) fetch(mi + 1, c ^ 1);
            const f32x4 part0 = mfma_k128(bg, a[c]), part1 = mfma_k128(bu, a[c]);
            // One combined scale per token row and K block (token scale x
            // weight scale), so each MFMA output needs a single FMA.
            const float sg = sa[c] * g, su = sa[c] * u;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              acc[mi][0][r] = fmaf(part0[r], sg, acc[mi][0][r]);
              acc[mi][1][r] = fmaf(part1[r], su, acc[mi][1][r]);
            }
          }
        }
        st = st == kRing - 1 ? 0 : st + 1;
      }

      // 128 columns: one whole scale group of the activations, so they are
      // quantised here (s = max(max |a|, 1e-10) / 448, q = rne(clamp(a / s)),
      // the rule gemm2_narrow_kernel applies, on the same bf16 values). The
      // fp8 rows are staged in the A stage of the last step, which no load
      // targets before the next item's first step writes them out.
#pragma unroll
      for (int mi = 0; mi < MI; ++mi) {
        float m = 0.f;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float a = act_and_mul<ACT>(bf16_round(acc[mi][0][r]), bf16_round(acc[mi][1][r]));
          acc[mi][0][r] = a;
          m = fmaxf(m, fabsf(a));
        }
        m = quad16_max(m);
        if (q == 0) s_m[wave][16 * mi + j] = m;
      }
      lds_barrier();  // s_m; and every wave is done with the last stage
      if (tid < 16 * MI) {
        float m = s_m[0][tid];
#pragma unroll
        for (int w = 1; w < NW; ++w) m = fmaxf(m, s_m[w][tid]);
        s_q[tid] = quant_scale(m);
      }
      lds_barrier();
      // A lane's four columns are one word of its row; the row's 16-byte
      // pieces are rotated as in the operand stages, so that the 16 rows of
      // a store spread over the banks.
      uint8_t* stg = s_a[st == 0 ? kRing - 1 : st - 1];
#pragma unroll
      for (int mi = 0; mi < MI; ++mi) {
        const int row = 16 * mi + j;
        const Quant qr(s_q[row]);
        const uint32_t w = fp8x4(qr(acc[mi][0][0]), qr(acc[mi][0][1]), qr(acc[mi][0][2]), qr(acc[mi][0][3]));
        *reinterpret_cast<uint32_t*>(stg + row * kRowB + ((wave ^ (row & 7)) << 4) + 4 * q) = w;
      }
    });
    out_cb = cb;
    out_c0 = cur.col * NC;
    out_rows = 16 * nmi;
    if (!more) break;
    cur = nxt;
    nxt = after;
    ++n;
    cb = nb;
    ao_cur = ao_nxt;
  }
  lds_barrier();
  copy_out(s_a[st == 0 ? kRing - 1 : st - 1]);
  // The last steps requested blocks that nothing reads: let them land before
  // the workgroup's LDS is released.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// Operands of one K block of a 16-row subtile for one wave: the A rows (the
// lane's row j, bytes 32q..32q+31) and two 16-row blocks of B rows.
struct KBlock {
  u32x4 a[2];
  u32x4 b[2][2];
};

// CH consecutive K blocks from kb0, the block index clamped at KB - 1 so
// that the loads are unconditional (a clamped block is loaded, not used).
// The weight rows (B) and the token rows (A) load separately, so that the
// weights can be requested before the tile's rows are looked up.
template <int CH>
__device__ __forceinline__ void load_chunk_b(KBlock (&c)[CH], const uint8_t* const (&brow)[2], int kb0, int KB) {
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    const int kb = kb0 + i < KB ? kb0 + i : KB - 1;
    load32(brow[0] + kb * kKB, c[i].b[0]);
    load32(brow[1] + kb * kKB, c[i].b[1]);
  }
}

template <int CH>
__device__ __forceinline__ void load_chunk_a(KBlock (&c)[CH], const uint8_t* arow, int kb0, int KB) {
#pragma unroll
  for (int i = 0; i < CH; ++i) load32(arow + (kb0 + i < KB ? kb0 + i : KB - 1) * kKB, c[i].a);
}

template <int CH>
__device__ __forceinline__ void load_chunk(KBlock (&c)[CH], const uint8_t* arow, const uint8_t* const (&brow)[2],
                                           int kb0, int KB) {
  load_chunk_b<CH>(c, brow, kb0, KB);
  load_chunk_a<CH>(c, arow, kb0, KB);
}

// The rows of one 16-row subtile (r0 = its first row in the tile): the
// pair of each row (-1 for padding) and the operand row it reads (padding
// repeats the subtile's first pair).
__device__ __forceinline__ void subtile_rows(const Tile& tile, int r0, const int32_t* pairs, int div, int* s_pair,
                                             int* s_row) {
  const int tid = threadIdx.x;
  if (tid < 16) {
    const int n = tile.count - r0;
    const int p = pairs[tile.first + r0 + (tid < n ? tid : 0)];
    s_pair[tid] = tid < n ? p : -1;
    s_row[tid] = p / div;
  }
}

// GEMM1 for small batches (decode): one 16-row subtile of a tile x 16
// activation columns (gate rows n and up rows I + n) per workgroup. A lone
// subtile is bound by load latency, so the 4 waves split each round of up to
// kSplitRound K blocks, issue all their loads at once and park the raw
// 16x16x128 products in LDS; wave 0 then scales them and sums them in K
// order with one FMA per block and output, the arithmetic of gemm1_kernel,
// so the bits do not depend on the split. 1-D grid in XCD order over
// (subtile, column block) items.
constexpr int kSplitRound = 16;  // K blocks per round, kSplitRound / 4 per wave

template <int ACT>
__global__ void __launch_bounds__(kThreads) gemm1_narrow_kernel(const uint8_t* __restrict__ xq,
                                                                const float* __restrict__ xs, int64_t H, int64_t I,
                                                                int topk, const uint8_t* __restrict__ w13,
                                                                const float* __restrict__ w13_scale,
                                                                const int32_t* __restrict__ offsets,
                                                                const int32_t* __restrict__ pairs,
                                                                const int32_t* __restrict__ tiles, int nsub,
                                                                Work work) {
  constexpr int kPerWave = kSplitRound / (kThreads / 64);
  __shared__ int s_row[16];
  __shared__ int s_pair[16];
  __shared__ float s_xs[16 * kMaxKB];
  __shared__ float s_sw[2][kMaxKB];
  __shared__ float s_m[16];
  __shared__ f32x4 s_part[kSplitRound][2][64];
  __shared__ __attribute__((aligned(16))) uint16_t s_o[16 * 16];

  const int ncb = static_cast<int>(I / 16);
  Tile tile;
  int ti, item;
  xcd_item(nsub * ncb, ti, item);
  if (!load_tile_at(ti, tiles, offsets, tile)) return;
  const int sub = item / ncb, r0 = 16 * sub;
  if (r0 >= tile.count) return;
  const int c0 = (item - sub * ncb) * 16;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int q = lane >> 4, j = lane & 15;
  const int KB = static_cast<int>(H / kKB);

  // The first round's weight rows depend on the slot alone: request them
  // before the rows and scales are looked up.
  const uint8_t* wslot = w13 + static_cast<int64_t>(tile.slot) * 2 * I * H;
  const int64_t n = c0 + j;
  const uint8_t* const brow[2] = {wslot + n * H + 32 * q, wslot + (I + n) * H + 32 * q};
  const int kw0 = wave * kPerWave;  // this wave's first block of each round, less the round's start
  KBlock c[kPerWave];
  load_chunk_b<kPerWave>(c, brow, kw0, KB);

  subtile_rows(tile, r0, pairs, topk, s_pair, s_row);
  __syncthreads();
  for (int i = tid; i < 16 * KB; i += kThreads) {
    const int r = i / KB, kb = i - r * KB;
    s_xs[i] = xs[static_cast<int64_t>(s_row[r]) * KB + kb];
  }
  {
    const float* sg = w13_scale + (static_cast<int64_t>(tile.slot) * (2 * I / kKB) + c0 / kKB) * KB;
    const float* su = w13_scale + (static_cast<int64_t>(tile.slot) * (2 * I / kKB) + (I + c0) / kKB) * KB;
    for (int i = tid; i < 2 * KB; i += kThreads) s_sw[i / KB][i % KB] = (i < KB ? sg : su)[i % KB];
  }
  const uint8_t* arow = xq + static_cast<int64_t>(s_row[j]) * H + 32 * q;
  load_chunk_a<kPerWave>(c, arow, kw0, KB);
  __syncthreads();  // s_xs, s_sw

  f32x4 acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};  // wave 0's sums
  for (int k0 = 0; k0 < KB; k0 += kSplitRound) {
    const int kw = k0 + kw0;  // this wave's first block of the round
    if (k0 > 0) load_chunk<kPerWave>(c, arow, brow, kw, KB);
#pragma unroll
    for (int i = 0; i < kPerWave; ++i) {
      if (kw + i >= KB) continue;
      s_part[wave * kPerWave + i][0][lane] = mfma_k128(c[i].a, c[i].b[0]);
      s_part[wave * kPerWave + i][1][lane] = mfma_k128(c[i].a, c[i].b[1]);
    }
    __syncthreads();
    if (wave == 0) {
      const int nk = KB - k0 < kSplitRound ? KB - k0 : kSplitRound;
      for (int t = 0; t < nk; ++t) {
        const int kb = k0 + t;
        const float g = s_sw[0][kb], u = s_sw[1][kb];
        const f32x4 pg = s_part[t][0][lane], pu = s_part[t][1][lane];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float sa = s_xs[(4 * q + r) * KB + kb];
          acc[0][r] = fmaf(pg[r], sa * g, acc[0][r]);
          acc[1][r] = fmaf(pu[r], sa * u, acc[1][r]);
        }
      }
    }
    __syncthreads();  // s_part is rewritten by the next round
  }

  if (wave == 0) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float a = act_and_mul<ACT>(bf16_round(acc[0][r]), bf16_round(acc[1][r]));
      float m = fabsf(a);
      m = row16_max(m);
      const int row = 4 * q + r;
      if (j == 0) s_m[row] = m;
      s_o[row * 16 + j] = static_cast<uint16_t>(bf16_bits(a));
    }
  }
  __syncthreads();
  if (tid < 16) {
    const int p = s_pair[tid];
    if (p >= 0) work.amax16[static_cast<int64_t>(p) * (I / 16) + c0 / 16] = s_m[tid];
  } else if (tid < 48) {  // 16 rows x 2 pieces of 16 bytes
    const int row = (tid - 16) >> 1, piece = tid & 1;
    const int p = s_pair[row];
    if (p >= 0)
      *reinterpret_cast<u32x4*>(work.a16 + static_cast<int64_t>(p) * I + c0 + piece * 8) =
          *reinterpret_cast<const u32x4*>(s_o + row * 16 + piece * 8);
  }
}

// ---- decode steps: two launches for the expert FFN ----
//
// For at most kDecodePairs pairs, every wave of every gemm1 workgroup routes
// the pairs itself (one pair per lane) and the workgroup quantises the token
// rows it multiplies into LDS, so no routing or quantisation launch precedes
// it. gemm2 then takes one token and 8 or 16 output columns per workgroup, computes
// each of the token's pairs and sums them there, so no top-k sum launch
// follows. The bits are those of xp_moe_quant_route, xp_moe_experts and
// xp_moe_topk_sum.
constexpr int kDecodePairs = 64;
constexpr int kDecodeMaxH = 4096;       // 16 quantised token rows of H bytes fit in LDS
constexpr int kDecodeActBytes = 32768;  // a token's quantised activations (topk x I) in LDS

// Pair p's slot (-1: an id outside [0, E) or an expert without a slot):
// from the acquire's per-pair slots when given, else ids then expert_map.
__device__ __forceinline__ int decode_slot(int p, int n, const void* ids, int eb, const int32_t* __restrict__ expert_map,
                                           const int32_t* __restrict__ pair_slot, int E, int slots) {
  const int pc = p < n ? p : 0;  // unconditional loads; lanes past n are not routed
  int sl;
  if (pair_slot) {
    sl = pair_slot[pc];
  } else {
    const int64_t e = load_id(ids, eb, pc);
    sl = e >= 0 && e < E ? expert_map[e] : -1;
  }
  return p < n && sl >= 0 && sl < slots ? sl : -1;
}

// The step's routing, computed by one wave from the pairs' slots (lane p:
// pair p): on the lane of each slot's first pair, the slot's ROWS-row subtiles
// (nsub) and the index of its first one among all the step's subtiles, in the
// order of the slots' first pairs (start); zero subtiles on the other lanes.
// The lanes of one slot are found bit by bit of the slot number, so the cost
// is the bits of `slots`, not the pairs: every wave of every workgroup routes,
// and readlane loops over 32 pairs took 3 us of a 4-token step's 21.
struct DecodeRoute {
  int start, nsub;
};

template <int ROWS>
__device__ __forceinline__ DecodeRoute decode_route(int slot, int slots) {
  unsigned long long same = __ballot(slot >= 0);
  const int bits = 32 - __clz(slots - 1);  // of slots 0 .. slots - 1
  for (int b = 0; b < bits; ++b) {
    const bool set = (slot >> b) & 1;
    const unsigned long long m = __ballot(set);
    same &= set ? m : ~m;
  }
  const int count = slot >= 0 ? __popcll(same) : 0;
  const bool first = slot >= 0 && lane_prefix(same) == 0;
  const int nsub = first ? (count + ROWS - 1) / ROWS : 0;
  int start = 0;
#pragma unroll
  for (int b = 0; (kDecodePairs / ROWS) >> b; ++b)
    start += static_cast<int>(lane_prefix(__ballot((nsub >> b) & 1))) << b;
  return DecodeRoute{start, nsub};
}

// gemm1_narrow_kernel over a decode step's pairs, with their routing and the
// quantisation of their token rows done here. Dynamic LDS: the fp8 token rows.
// Every wave routes the step itself (a pair per lane), so the weight rows of
// the workgroup's slot are requested as soon as the pairs' slots arrive; the
// token rows, requested before them (one or two tokens: before the slots),
// are quantised while the weights are in flight.
//
// A workgroup takes ROWS pairs of a slot (the product always has 16 rows;
// those past ROWS are not kept). A few tokens give a slot a few pairs at
// most, and the LDS of 16 rows (32 KB of token rows at H = 2048, 32 KB of
// products) let only two workgroups share a CU, so that a step of 4 tokens
// ran in two rounds of load latencies. 4 tokens, 32 of 256 experts 2048 x
// 512: 25 -> 21 us with 4 rows, 16 us with the shorter routing (67 MB of
// weights: 2.7 -> 4.2 TB/s).
template <int ACT, int ROWS>
__global__ void __launch_bounds__(kThreads) gemm1_decode_kernel(
    const uint16_t* __restrict__ x, int64_t H, int64_t I, const void* ids, int eb, int npairs, int topk,
    const int32_t* __restrict__ expert_map, const int32_t* __restrict__ pair_slot, int E, int slots,
    const uint8_t* __restrict__ w13,
    const float* __restrict__ w13_scale, Work work) {
  constexpr int kPerWave = kSplitRound / (kThreads / 64);
  constexpr int kPre = 4;  // token pieces per thread requested before the routing
  constexpr int kLanes = 4 * ROWS;  // lanes 16q + j whose product rows 4q .. 4q + 3 are below ROWS
  static_assert(ROWS == 4 || ROWS == 8 || ROWS == 16, "whole 4-row groups of the product");
  extern __shared__ __attribute__((aligned(16))) uint8_t s_aq[];  // [rows][H] fp8 token rows
  __shared__ int s_pair[ROWS];
  __shared__ int s_arow[16];             // LDS row of each product row's activations
  __shared__ float s_xs[ROWS * kMaxKB];  // their scales [LDS row][K block]
  __shared__ float s_sw[2][kMaxKB];
  __shared__ float s_m[ROWS];
  // Raw products of a round: [K block][gate, up][row within the lane's
  // 4-row group][lane], so that a wave reads its own row's values in lane
  // order.
  __shared__ float s_part[kSplitRound][2][4][kLanes];
  __shared__ __attribute__((aligned(16))) uint16_t s_o[ROWS * 16];

  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int q = lane >> 4, j = lane & 15;
  const int KB = static_cast<int>(H / kKB);

  // A token piece (8 columns of token t from column c8) quantised as
  // quant_tokens_kernel does (16 lanes per 128-column group) into LDS row r.
  auto quant_piece = [&](const u32x4& raw, int r, int c8) {
    float v[8];
    float amax = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[2 * i] = bf16_value(raw[i] & 0xffffu);
      v[2 * i + 1] = bf16_value(raw[i] >> 16);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) amax = fmaxf(amax, fabsf(v[i]));
    amax = row16_max(amax);
    const float sc = quant_scale(amax);
    *reinterpret_cast<uint2*>(s_aq + r * H + c8) = quant_words(raw, sc);
    if ((tid & 15) == 0) s_xs[r * KB + c8 / kKB] = sc;
  };
  // With one or two tokens, all their rows are requested before the routing
  // and quantised (piece i of the step: token i / (H / 8)): a batch-1 step
  // is bound by load latency. With more, each workgroup quantises only its
  // subtile's rows once they are known (its pairs are mostly of different
  // tokens, and every token row of the step would be quantised in each of
  // hundreds of workgroups: 143 against 31 us at 8 tokens).
  const int ntok = npairs / topk;
  const bool by_token = ntok <= 2;
  const int nc8 = static_cast<int>(H / 8);
  int npiece = by_token ? ntok * nc8 : 0;
  auto piece_ptr = [&](int i) { return x + static_cast<int64_t>(i / nc8) * H + (i % nc8) * 8; };
  u32x4 xr[kPre];
  if (by_token) {
#pragma unroll
    for (int i = 0; i < kPre; ++i) {
      const int it = tid + kThreads * i;
      xr[i] = *reinterpret_cast<const u32x4*>(piece_ptr(it < npiece ? it : 0));
    }
  }

  const int slot_l = decode_slot(lane, npairs, ids, eb, expert_map, pair_slot, E, slots);
  // gemm2_decode_kernel reads the pairs' slots from the workspace (the
  // activation-scale region, which the decode path does not use).
  if (blockIdx.x == 0 && wave == 0 && lane < npairs) reinterpret_cast<int32_t*>(work.acts)[lane] = slot_l;
  const DecodeRoute rt = decode_route<ROWS>(slot_l, slots);

  // The workgroup's subtile among all the step's and its column block; the grid bounds the subtiles (the same in every wave).
  const int ncb = static_cast<int>(I / 16);
  int gsi, cbk;
  xcd_item(ncb, gsi, cbk);
  const unsigned long long own = __ballot(rt.nsub > 0 && rt.start <= gsi && gsi < rt.start + rt.nsub);
  if (own == 0) return;
  const int lead = __ffsll(static_cast<long long>(own)) - 1;
  const int slot = __builtin_amdgcn_readlane(slot_l, lead);
  const int sub = gsi - __builtin_amdgcn_readlane(rt.start, lead);
  const unsigned long long mine = __ballot(slot_l == slot);
  const int count = __popcll(mine);
  const int r0 = ROWS * sub;  // below count
  const int c0 = cbk * 16;
  const int nrow = count - r0 < ROWS ? count - r0 : ROWS;
  // The subtile's rows: the slot's pairs in pair order, rows r0 .. r0 + nrow
  // - 1; row r's pair goes to lane r (and lane 63 takes the other lanes').
  const int rk = static_cast<int>(lane_prefix(mine)) - r0;
  const bool in_sub = slot_l == slot && rk >= 0 && rk < ROWS;
  const int row_pair = __builtin_amdgcn_ds_permute(4 * (in_sub ? rk : 63), lane);
  if (!by_token) {
    npiece = nrow * nc8;
#pragma unroll
    for (int i = 0; i < kPre; ++i) {
      const int it = tid + kThreads * i < npiece ? tid + kThreads * i : 0;
      const int r = it / nc8, p = __builtin_amdgcn_ds_bpermute(4 * r, row_pair);
      xr[i] = *reinterpret_cast<const u32x4*>(x + static_cast<int64_t>(p / topk) * H + (it - r * nc8) * 8);
    }
  }

  // The slot's gate and up scales, then its weight rows, requested at once.
  const float* sg = w13_scale + (static_cast<int64_t>(slot) * (2 * I / kKB) + c0 / kKB) * KB;
  const float* su = w13_scale + (static_cast<int64_t>(slot) * (2 * I / kKB) + (I + c0) / kKB) * KB;
  const int si = tid < 2 * KB ? tid : 0;
  const float sw = (si < KB ? sg : su)[si < KB ? si : si - KB];
  const uint8_t* wslot = w13 + static_cast<int64_t>(slot) * 2 * I * H;
  const int64_t n = c0 + j;
  const uint8_t* const brow[2] = {wslot + n * H + 32 * q, wslot + (I + n) * H + 32 * q};
  const int kw0 = wave * kPerWave;
  KBlock c[kPerWave];
  load_chunk_b<kPerWave>(c, brow, kw0, KB);

  // Token rows into LDS while the weights are in flight: all of them, or the
  // subtile's.
#pragma unroll
  for (int i = 0; i < kPre; ++i) {
    const int it = tid + kThreads * i;
    if (it < npiece) quant_piece(xr[i], it / nc8, (it % nc8) * 8);  // whole 16-lane groups
  }
  for (int it0 = kThreads * kPre; it0 < npiece; it0 += kThreads) {
    const int it = it0 + tid < npiece ? it0 + tid : 0, r = it / nc8;
    const int p = __builtin_amdgcn_ds_bpermute(4 * r, row_pair);
    const int64_t t = by_token ? r : p / topk;
    const u32x4 raw = *reinterpret_cast<const u32x4*>(x + t * H + (it - r * nc8) * 8);
    if (it0 + tid < npiece) quant_piece(raw, r, (it - r * nc8) * 8);
  }
  if (tid < 2 * KB) s_sw[tid / KB][tid % KB] = sw;
  // Rows past nrow (outputs not stored) read the subtile's first row.
  if (tid < 16) {
    if (tid < ROWS) s_pair[tid] = tid < nrow ? row_pair : -1;
    const int first = __builtin_amdgcn_readlane(row_pair, 0);
    s_arow[tid] = by_token ? (tid < nrow ? row_pair : first) / topk : (tid < nrow ? tid : 0);
  }
  __syncthreads();  // s_aq, s_xs, s_sw, s_pair, s_arow

  const uint8_t* arow = s_aq + s_arow[j] * H + 32 * q;
  auto load_a = [&](int kb0) {
#pragma unroll
    for (int i = 0; i < kPerWave; ++i) {
      const int kb = kb0 + i < KB ? kb0 + i : KB - 1;
      c[i].a[0] = *reinterpret_cast<const u32x4*>(arow + kb * kKB);
      c[i].a[1] = *reinterpret_cast<const u32x4*>(arow + kb * kKB + 16);
    }
  };
  // Wave w scales and sums row 4q + w of the lane's 4-row group (gate and
  // up) in K order, one FMA per block, as gemm1_kernel does.
  // The lanes past kLanes repeat the others'.
  const int sl = lane & (kLanes - 1);
  const int row = 4 * (sl >> 4) + wave;
  const int ar = s_arow[row];
  float acc_g = 0.f, acc_u = 0.f;
  for (int k0 = 0; k0 < KB; k0 += kSplitRound) {
    const int kw = k0 + kw0;
    if (k0 > 0) load_chunk_b<kPerWave>(c, brow, kw, KB);
    load_a(kw);
#pragma unroll
    for (int i = 0; i < kPerWave; ++i) {
      if (kw + i >= KB) continue;
      const f32x4 pg = mfma_k128(c[i].a, c[i].b[0]), pu = mfma_k128(c[i].a, c[i].b[1]);
      if (lane >= kLanes) continue;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        s_part[wave * kPerWave + i][0][r][lane] = pg[r];
        s_part[wave * kPerWave + i][1][r][lane] = pu[r];
      }
    }
    __syncthreads();
    // Row `wave` of the lane's group: fixed offsets from one address, and
    // the whole round unrolled, so every LDS read of the sum is in flight
    // before the FMAs that consume it.
    const float* sp = &s_part[0][0][wave][sl];
    const float* sx = s_xs + ar * KB + k0;
    auto sum_block = [&](int t) {
      const float sa = sx[t];
      acc_g = fmaf(sp[(2 * t) * 4 * kLanes], sa * s_sw[0][k0 + t], acc_g);
      acc_u = fmaf(sp[(2 * t + 1) * 4 * kLanes], sa * s_sw[1][k0 + t], acc_u);
    };
    if (KB - k0 >= kSplitRound) {
#pragma unroll
      for (int t = 0; t < kSplitRound; ++t) sum_block(t);
    } else {
      for (int t = 0; t < KB - k0; ++t) sum_block(t);
    }
    __syncthreads();  // s_part is rewritten by the next round
  }

  {
    const float a = act_and_mul<ACT>(bf16_round(acc_g), bf16_round(acc_u));
    const float m = row16_max(fabsf(a));
    if (j == 0) s_m[row] = m;
    s_o[row * 16 + j] = static_cast<uint16_t>(bf16_bits(a));
  }
  __syncthreads();
  if (tid < ROWS) {
    const int p = s_pair[tid];
    if (p >= 0) work.amax16[static_cast<int64_t>(p) * (I / 16) + c0 / 16] = s_m[tid];
  } else if (tid >= 16 && tid < 16 + 2 * ROWS) {  // ROWS rows x 2 pieces of 16 bytes
    const int rr = (tid - 16) >> 1, piece = tid & 1;
    const int p = s_pair[rr];
    if (p >= 0)
      *reinterpret_cast<u32x4*>(work.a16 + static_cast<int64_t>(p) * I + c0 + piece * 8) =
          *reinterpret_cast<const u32x4*>(s_o + rr * 16 + piece * 8);
  }
}

// gemm2 of a decode step with the top-k sum: one workgroup per token and COLS
// output columns. A single token takes 8, so that its weight rows spread over
// 256 workgroups at H = 2048; then lanes j and j + 8 of the MFMA operand read
// the same row (one request), and columns 8-15 of the product are not used.
// More tokens fill the GPU with 16 columns, and half as many workgroups
// quantise each token's activations (4 tokens, 32 experts 2048 x 512: 13.1 ->
// 9.2 us; the quantisation was the larger part of a workgroup's
// instructions). Its waves take the token's pairs two at a time (wave w:
// pairs w and w + 4, then w + 8 and w + 12, ...); each pair's contributions
// are computed as gemm2_narrow_kernel computes them (the token's quantised
// activation row as every row of the MFMA operand, kNarrowChunk K blocks of
// weight rows per load) and rounded to bf16; then the contributions are
// summed in k order in fp32 and rounded once, as topk_sum_kernel does. A
// token's experts are distinct slots, so its pairs share no weights. The
// pairs' slots come from gemm1_decode_kernel's routing through the workspace,
// one load instead of the ids and expert_map lookups. Pairs whose id is
// outside [0, E) add nothing; so do pairs without a slot (the separate calls
// would read a contribution never written). The slots, the routed weights and
// the first activation pieces are requested first, then each wave's first two
// pairs' weight rows, and the activations are quantised while those are in
// flight.
template <int COLS>
__global__ void __launch_bounds__(kThreads) gemm2_decode_kernel(
    int64_t H, int64_t I, int topk, const float* __restrict__ topk_weight, const uint8_t* __restrict__ w2,
    const float* __restrict__ w2_scale, Work work, uint16_t* __restrict__ out) {
  constexpr int NWAVE = kThreads / 64;
  constexpr int kPre = 2;  // activation pieces per thread requested before the weights
  extern __shared__ __attribute__((aligned(16))) uint8_t s_act[];  // [topk][I] fp8 activations
  __shared__ int s_slot[kDecodePairs];
  __shared__ float s_as[kDecodePairs * 4];  // activation scales [pair][K block], K blocks of a round
  __shared__ uint16_t s_c[kDecodePairs][COLS];

  const int ncol = static_cast<int>(H / COLS);
  const int t = static_cast<int>(blockIdx.x) / ncol;
  const int n0 = (static_cast<int>(blockIdx.x) - t * ncol) * COLS;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int q = lane >> 4, j = lane & 15;
  const int KB = static_cast<int>(I / kKB);
  const int64_t p0 = static_cast<int64_t>(t) * topk;
  const int nc8 = static_cast<int>(I / 8), npiece = topk * nc8;

  // Requests: the pairs' slots as gemm1_decode_kernel routed them (-1: an
  // invalid id or an expert without a slot), the wave's first two pairs'
  // slots and routed weights, and the first activation pieces (8 columns of
  // pair k's bf16 row with the eight 16-column maxima of its group).
  const int32_t* pslot = reinterpret_cast<const int32_t*>(work.acts) + p0;
  const int my_slot = pslot[tid < topk ? tid : 0];
  int kk0[2] = {wave, wave + NWAVE};
  int slot0[2];
  float tw0[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int kc = kk0[h] < topk ? kk0[h] : 0;
    slot0[h] = pslot[kc];
    tw0[h] = topk_weight[p0 + kc];
  }
  auto piece_at = [&](int it, int& k, int& c8) {
    k = it / nc8;
    c8 = (it - k * nc8) * 8;
  };
  u32x4 av[kPre], am[kPre][2];
#pragma unroll
  for (int i = 0; i < kPre; ++i) {
    const int it = tid + kThreads * i;
    int k, c8;
    piece_at(it < npiece ? it : 0, k, c8);
    const int64_t p = p0 + k;
    av[i] = *reinterpret_cast<const u32x4*>(work.a16 + p * I + c8);
    const float* m = work.amax16 + p * (I / 16) + 8 * (c8 / kKB);
    am[i][0] = *reinterpret_cast<const u32x4*>(m);
    am[i][1] = *reinterpret_cast<const u32x4*>(m + 4);
  }

  // A pair's weight rows for output columns n0 .. n0 + COLS - 1 and their scales.
  auto pair_rows = [&](int slot, const uint8_t*& brow, const float*& sw) {
    const int sl = slot < 0 ? 0 : slot;
    brow = w2 + static_cast<int64_t>(sl) * H * I + static_cast<int64_t>(n0 + (j & (COLS - 1))) * I + 32 * q;
    sw = w2_scale + (static_cast<int64_t>(sl) * (H / kKB) + n0 / kKB) * KB;
  };
  // A chunk's weight rows of two pairs, with their K blocks' scales.
  auto load_rows = [&](const int (&slot)[2], const uint8_t* const (&brow)[2], const float* const (&sw)[2], int k0,
                       u32x4 (&b)[2][kNarrowChunk][2], float (&wsc)[2][kNarrowChunk]) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (slot[h] < 0) continue;  // uniform
#pragma unroll
      for (int i = 0; i < kNarrowChunk; ++i) {
        const int kb = k0 + i < KB ? k0 + i : KB - 1;
        wsc[h][i] = sw[h][kb];
        load32(brow[h] + kb * kKB, b[h][i]);
      }
    }
  };
#pragma unroll
  for (int h = 0; h < 2; ++h) slot0[h] = kk0[h] < topk ? slot0[h] : -1;
  const uint8_t* brow0[2];
  const float* sw0[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) pair_rows(slot0[h], brow0[h], sw0[h]);
  u32x4 b0[2][kNarrowChunk][2];
  float wsc0[2][kNarrowChunk];
  load_rows(slot0, brow0, sw0, 0, b0, wsc0);

  // The activations quantised into LDS as gemm2_narrow_kernel quantises them
  // (a 128-column group's scale from its eight 16-column maxima).
  auto quant_piece = [&](const u32x4& v, const u32x4 (&mm)[2], int it) {
    int k, c8;
    piece_at(it, k, c8);
    const int g = c8 / kKB;
    float mx = __uint_as_float(mm[0][0]);
#pragma unroll
    for (int u = 1; u < 4; ++u) mx = fmaxf(mx, __uint_as_float(mm[0][u]));
#pragma unroll
    for (int u = 0; u < 4; ++u) mx = fmaxf(mx, __uint_as_float(mm[1][u]));
    const float sc = quant_scale(mx);
    if (c8 % kKB == 0 && g < 4) s_as[k * 4 + g] = sc;
    *reinterpret_cast<uint2*>(s_act + k * I + c8) = quant_words(v, sc);
  };
  if (tid < topk) s_slot[tid] = my_slot;
#pragma unroll
  for (int i = 0; i < kPre; ++i) {
    const int it = tid + kThreads * i;
    if (it < npiece) quant_piece(av[i], am[i], it);
  }
  for (int it = tid + kThreads * kPre; it < npiece; it += kThreads) {
    int k, c8;
    piece_at(it, k, c8);
    const int64_t p = p0 + k;
    const float* m = work.amax16 + p * (I / 16) + 8 * (c8 / kKB);
    const u32x4 mm[2] = {*reinterpret_cast<const u32x4*>(m), *reinterpret_cast<const u32x4*>(m + 4)};
    quant_piece(*reinterpret_cast<const u32x4*>(work.a16 + p * I + c8), mm, it);
  }
  __syncthreads();

  // One chunk of K blocks of two pairs: their 16 columns scaled and summed
  // in K order in fp32 (row 0 of the product, lanes q = 0, is the pair's
  // value).
  auto mul_chunk = [&](const u32x4 (&b)[2][kNarrowChunk][2], const float (&wsc)[2][kNarrowChunk],
                       const int (&kk)[2], const int (&slot)[2], int k0, float (&acc)[2]) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (slot[h] < 0) continue;
      const int64_t p = p0 + kk[h];
      const uint8_t* arow = s_act + kk[h] * I + 32 * q;
      if (k0 + kNarrowChunk <= KB && k0 + kNarrowChunk <= 4) {
        // A whole chunk whose activation scales are all in LDS: every LDS
        // read first, then the products, in K order.
        u32x4 a[kNarrowChunk][2];
        float sa[kNarrowChunk];
#pragma unroll
        for (int i = 0; i < kNarrowChunk; ++i) {
          a[i][0] = *reinterpret_cast<const u32x4*>(arow + (k0 + i) * kKB);
          a[i][1] = *reinterpret_cast<const u32x4*>(arow + (k0 + i) * kKB + 16);
          sa[i] = s_as[kk[h] * 4 + k0 + i];
        }
#pragma unroll
        for (int i = 0; i < kNarrowChunk; ++i) {
          const f32x4 part = mfma_k128(a[i], b[h][i]);
          acc[h] = fmaf(part[0], sa[i] * wsc[h][i], acc[h]);
        }
        continue;
      }
#pragma unroll
      for (int i = 0; i < kNarrowChunk; ++i) {
        const int kb = k0 + i;
        if (kb >= KB) continue;
        u32x4 a[2];
        a[0] = *reinterpret_cast<const u32x4*>(arow + kb * kKB);
        a[1] = *reinterpret_cast<const u32x4*>(arow + kb * kKB + 16);
        // the pair's activation scale for this K block: from LDS for the
        // first four blocks, else recomputed from the maxima
        float sa;
        if (kb < 4) {
          sa = s_as[kk[h] * 4 + kb];
        } else {
          const float* m = work.amax16 + p * (I / 16) + 8 * kb;
          float mx = m[0];
#pragma unroll
          for (int u = 1; u < 8; ++u) mx = fmaxf(mx, m[u]);
          sa = quant_scale(mx);
        }
        const f32x4 part = mfma_k128(a, b[h][i]);
        acc[h] = fmaf(part[0], sa * wsc[h][i], acc[h]);
      }
    }
  };
  auto finish = [&](const int (&kk)[2], const int (&slot)[2], const float (&acc)[2], const float (&tw)[2]) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (kk[h] >= topk || q != 0 || j >= COLS) continue;
      s_c[kk[h]][j] = slot[h] < 0 ? 0 : static_cast<uint16_t>(bf16_bits(acc[h] * tw[h]));
    }
  };

  // The wave's first two pairs, their first chunk already loaded.
  {
    float acc[2] = {0.f, 0.f};
    mul_chunk(b0, wsc0, kk0, slot0, 0, acc);
    for (int k0 = kNarrowChunk; k0 < KB; k0 += kNarrowChunk) {
      u32x4 b[2][kNarrowChunk][2];
      float wsc[2][kNarrowChunk];
      load_rows(slot0, brow0, sw0, k0, b, wsc);
      mul_chunk(b, wsc, kk0, slot0, k0, acc);
    }
    finish(kk0, slot0, acc, tw0);
  }
  // Further pairs (top-k above 2 x 4 waves), two at a time.
  for (int k = wave + 2 * NWAVE; k < topk; k += 2 * NWAVE) {
    const int kk[2] = {k, k + NWAVE};
    int slot[2];
    float tw[2];
    const uint8_t* brow[2];
    const float* sw[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      slot[h] = kk[h] < topk ? s_slot[kk[h]] : -1;
      tw[h] = kk[h] < topk ? topk_weight[p0 + kk[h]] : 0.f;
      pair_rows(slot[h], brow[h], sw[h]);
    }
    float acc[2] = {0.f, 0.f};
    for (int k0 = 0; k0 < KB; k0 += kNarrowChunk) {
      u32x4 b[2][kNarrowChunk][2];
      float wsc[2][kNarrowChunk];
      load_rows(slot, brow, sw, k0, b, wsc);
      mul_chunk(b, wsc, kk, slot, k0, acc);
    }
    finish(kk, slot, acc, tw);
  }
  __syncthreads();
  if (tid < COLS) {
    // The token's contributions in k order, eight LDS reads in flight at a
    // time.
    float sum = 0.f;
    for (int k0 = 0; k0 < topk; k0 += 8) {
      int sl[8];
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int k = k0 + u < topk ? k0 + u : topk - 1;
        sl[u] = s_slot[k];
        v[u] = bf16_value(s_c[k][tid]);
      }
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (k0 + u < topk && sl[u] >= 0) sum += v[u];
    }
    out[static_cast<int64_t>(t) * H + n0 + tid] = static_cast<uint16_t>(bf16_bits(sum));
  }
}

// GEMM2 for small batches: one 16-row subtile x 128 output columns (4 waves
// x 32). The subtile's activations arrive as bf16 rows with their
// 16-column maxima (gemm1_narrow_kernel's output): the workgroup quantises
// them itself, with the rule gemm1_kernel applies at prefill sizes, into
// LDS, kQuantK columns per round, and multiplies them from there; the
// weight rows come straight from global memory, CH K blocks per load chunk
// (the first chunk requested before the rows are looked up). Same sums and
// rounding as gemm2_kernel.
constexpr int kQuantK = 2048;  // activation columns quantised per LDS round

template <int CH>
__global__ void __launch_bounds__(kThreads) gemm2_narrow_kernel(int64_t H, int64_t I,
                                                                const float* __restrict__ topk_weight,
                                                                const uint8_t* __restrict__ w2,
                                                                const float* __restrict__ w2_scale,
                                                                const int32_t* __restrict__ offsets,
                                                                const int32_t* __restrict__ pairs,
                                                                const int32_t* __restrict__ tiles, int nsub,
                                                                Work work, uint16_t* __restrict__ out) {
  constexpr int kRoundKB = kQuantK / kKB;
  __shared__ int s_row[16];
  __shared__ int s_pair[16];
  __shared__ float s_as[16 * kMaxKB];
  __shared__ float s_w[16];
  __shared__ float s_sw[kMaxKB];
  __shared__ __attribute__((aligned(16))) uint8_t s_act[16 * kQuantK];
  __shared__ __attribute__((aligned(16))) uint16_t s_o[16 * kBN];

  const int ncb = static_cast<int>(H / kBN);
  Tile tile;
  int ti, item;
  xcd_item(nsub * ncb, ti, item);
  const int sub = item / ncb, cb = item - sub * ncb;
  if (!load_tile_at(ti, tiles, offsets, tile)) return;
  const int r0 = 16 * sub;
  if (r0 >= tile.count) return;
  const int n0 = cb * kBN;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int q = lane >> 4, j = lane & 15;
  const int KB = static_cast<int>(I / kKB);

  // Weight rows of the first chunk first: they depend on the slot alone.
  const uint8_t* wslot = w2 + static_cast<int64_t>(tile.slot) * H * I;
  const uint8_t* const brow[2] = {wslot + static_cast<int64_t>(n0 + 32 * wave + j) * I + 32 * q,
                                  wslot + static_cast<int64_t>(n0 + 32 * wave + 16 + j) * I + 32 * q};
  KBlock c[CH];
  load_chunk_b<CH>(c, brow, 0, KB);

  subtile_rows(tile, r0, pairs, 1, s_pair, s_row);
  __syncthreads();
  if (tid < 16) s_w[tid] = s_pair[tid] >= 0 ? topk_weight[s_pair[tid]] : 0.f;
  if (tid < KB) s_sw[tid] = w2_scale[(static_cast<int64_t>(tile.slot) * (H / kKB) + n0 / kKB) * KB + tid];

  f32x4 acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
  for (int k0 = 0; k0 < KB; k0 += kRoundKB) {
    const int nk = KB - k0 < kRoundKB ? KB - k0 : kRoundKB;
    // Quantise columns [128 k0, 128 (k0 + nk)) of the 16 rows: per row and
    // 128-column group s = max(max |a|, 1e-10) / 448 from the eight
    // 16-column maxima, q = rne(clamp(a / s)); 8 columns per item.
    const int per_row = nk * (kKB / 8);
    for (int i = tid; i < 16 * per_row; i += kThreads) {
      const int r = i / per_row, c8 = (i - r * per_row) * 8, g = k0 + c8 / kKB;
      const int64_t p = s_row[r];
      const float* m = work.amax16 + p * (I / 16) + 8 * g;
      const u32x4 v = *reinterpret_cast<const u32x4*>(work.a16 + p * I + kKB * k0 + c8);
      float mx = m[0];
#pragma unroll
      for (int k = 1; k < 8; ++k) mx = fmaxf(mx, m[k]);
      const float sc = quant_scale(mx);
      if (c8 % kKB == 0) s_as[r * KB + g] = sc;
      *reinterpret_cast<uint2*>(s_act + r * kQuantK + c8) = quant_words(v, sc);
    }
    __syncthreads();  // s_act, s_as (and s_w, s_sw)
    for (int kc = 0; kc < nk; kc += CH) {
      if (k0 + kc > 0) load_chunk_b<CH>(c, brow, k0 + kc, KB);
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        const int kb = k0 + kc + i;
        if (kc + i >= nk) continue;
        const u32x4* pa = reinterpret_cast<const u32x4*>(s_act + j * kQuantK + (kb - k0) * kKB + 32 * q);
        const u32x4 a[2] = {pa[0], pa[1]};
        const float w = s_sw[kb];
        float sc[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) sc[r] = s_as[(4 * q + r) * KB + kb] * w;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const f32x4 part = mfma_k128(a, c[i].b[t]);
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[t][r] = fmaf(part[r], sc[r], acc[t][r]);
        }
      }
    }
    __syncthreads();  // the next round rewrites s_act
  }

#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = 4 * q + r;
    const float wgt = s_w[row];
#pragma unroll
    for (int t = 0; t < 2; ++t) s_o[row * kBN + 32 * wave + 16 * t + j] = static_cast<uint16_t>(bf16_bits(acc[t][r] * wgt));
  }
  __syncthreads();
  {  // 16 rows x 16 pieces of 16 bytes: one pass of the 256 threads
    const int row = tid >> 4, col = (tid & 15) * 8;
    const int p = s_pair[row];
    if (p >= 0)
      *reinterpret_cast<u32x4*>(out + static_cast<int64_t>(p) * H + n0 + col) =
          *reinterpret_cast<const u32x4*>(s_o + row * kBN + col);
  }
}

// GEMM2 at prefill sizes: down projection of 128 TB output columns of a wide
// tile per item, times the routed weight, bf16 rows per pair. Each of the 8
// waves owns 16 TB columns and runs the K blocks in order over the tile's
// fp8 activations; persistent over items through the operand ring as
// gemm1_kernel.
template <int TB, bool STREAM>
__global__ void __launch_bounds__(kGemmWaves * 64) gemm2_kernel(int64_t H, int64_t I,
                                                               const float* __restrict__ topk_weight,
                                                               const uint8_t* __restrict__ w2,
                                                               const float* __restrict__ w2_scale,
                                                               const int32_t* __restrict__ pairs,
                                                               const int32_t* __restrict__ wide, int64_t wmax,
                                                               int64_t npairs, Work work, uint16_t* __restrict__ out) {
  constexpr int NW = kGemmWaves, NT = NW * 64, NC = NW * 16 * TB;  // output columns per item
  constexpr int kStageRows = 64;  // output rows staged per epilogue round: 64 x NC bf16 = one weight stage
  static_assert(kStageRows * NC * 2 == NC * kRowB, "an epilogue round fills one weight stage");
  __shared__ __attribute__((aligned(16))) uint8_t s_b[kRing][NC * kRowB];
  __shared__ __attribute__((aligned(16))) uint8_t s_a[kRing][kWM * kRowB];
  __shared__ __attribute__((aligned(16))) float s_s[kRing][kWM];
  __shared__ int s_pn[kWM];
  __shared__ int s_row[2][kWM];
  __shared__ int s_pair[2][kWM];
  __shared__ float s_w[2][kWM];
  __shared__ float s_sw[2][2 * kMaxKB];  // weight scales per 128-row block (of TB) and K block, two items

  const int ncols = static_cast<int>(H / NC);
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int q = lane >> 4, j = lane & 15;
  const int KB = static_cast<int>(I / kKB), KS = KB > kMinSteps ? KB : kMinSteps;

  Item cur = item_fetch<STREAM>(0, ncols, wide, wmax);
  if (cur.count == 0) return;
  Item nxt = item_fetch<STREAM>(1, ncols, wide, wmax);
  int n = 2;

  // Weight-row loads: load i of a wave covers its stage rows 8i .. 8i + 7,
  // output columns 16 TB wave + 8i + lane / 8 of the item.
  uint32_t boff[2 * TB];
#pragma unroll
  for (int i = 0; i < 2 * TB; ++i)
    boff[i] = static_cast<uint32_t>((16 * TB * wave + 8 * i + (lane >> 3)) * I + 16 * swizzled_piece(lane));
  auto wbase = [&](const Item& it) {
    return w2 + (static_cast<int64_t>(it.slot) * H + static_cast<int64_t>(it.col) * NC) * I;
  };
  // Weight scales (TB 128-row blocks of w2 x KB) and routed weights of an
  // item into LDS, by waves 0 and 1; the rows s_row must be in place.
  auto request_scales = [&](const Item& it, const int* rows, float* sw, float* wt) {
    if (wave < 2) {
      const int i = tid < TB * KB ? tid : TB * KB - 1;
      const int t = i / KB, kb = i - t * KB;
      dma4(w2_scale, static_cast<uint32_t>(4 * ((static_cast<int64_t>(it.slot) * (H / kKB) + it.col * TB + t) * KB + kb)),
           sw + 64 * wave);
      dma4(topk_weight, static_cast<uint32_t>(4 * rows[tid]), wt + 64 * wave);
    }
  };
  // As gemm1_kernel's: the weight rows always, the A rows of live
  // subtiles, the A scales by waves 0 and 1; returns the loads issued.
  auto issue = [&](int stage, const uint8_t* wb, const AOffsets& ao, int kb, int nmi) {
    const uint8_t* bsrc = wb + kb * kRowB;
#pragma unroll
    for (int i = 0; i < 2 * TB; ++i) dma_weights<STREAM>(bsrc, boff[i], s_b[stage] + (16 * TB * wave + 8 * i) * kRowB);
    int ops = 2 * TB;
    if (wave < nmi) {
      const uint8_t* asrc = work.act + kb * kRowB;
#pragma unroll
      for (int i = 0; i < 2; ++i) dma16(asrc, ao.a[i], s_a[stage] + (16 * wave + 8 * i) * kRowB);
      ops += 2;
    }
    if (wave == 0 || (wave == 1 && nmi > 4)) {
      dma4(work.acts + kb, ao.s, &s_s[stage][64 * wave]);
      ops += 1;
    }
    return ops;
  };
  // Output rows [r0, r0 + rows) of an item, staged in LDS.
  int out_cb = 0, out_n0 = 0, out_r0 = 0, out_rows = 0;
  auto copy_out = [&](const uint16_t* stg) {
    for (int i = tid; i < out_rows * (NC / 8); i += NT) {
      const int rr = i / (NC / 8), piece = i - rr * (NC / 8);
      const int p = s_pair[out_cb][out_r0 + rr];
      *reinterpret_cast<u32x4*>(out + static_cast<int64_t>(p) * H + out_n0 + piece * 8) =
          *reinterpret_cast<const u32x4*>(stg + rr * NC + (piece ^ (rr & 15)) * 8);
    }
  };

  request_pairs(cur, pairs, s_pn);
  ring_barrier<0>();
  put_rows(cur, s_pn, 1, npairs, s_pair[0], s_row[0]);
  lds_barrier();
  request_scales(cur, s_row[0], s_sw[0], s_w[0]);
  AOffsets ao_cur = a_offsets(s_row[0], I, KB), ao_nxt = ao_cur;
  ring_barrier<0>();
  issue(0, wbase(cur), ao_cur, 0, (cur.count + 15) >> 4);
  int last_ops = issue(1, wbase(cur), ao_cur, KB > 1 ? 1 : 0, (cur.count + 15) >> 4);

  int st = 0;
  int cb = 0;
  for (;;) {
    const int nb = cb ^ 1;
    const bool more = nxt.count > 0;
    const uint8_t* wb_cur = wbase(cur);
    const uint8_t* wb_nxt = more ? wbase(nxt) : wb_cur;
    const int nmi = (cur.count + 15) >> 4, nmi_nxt = (nxt.count + 15) >> 4;
    const int n0 = cur.col * NC;
    Item after = nxt;

    with_subtiles(nmi, [&](auto nmi_c) {
      constexpr int MI = decltype(nmi_c)::value;
      f32x4 acc[MI][TB];
#pragma unroll
      for (int mi = 0; mi < MI; ++mi)
#pragma unroll
        for (int t = 0; t < TB; ++t) acc[mi][t] = f32x4{0.f, 0.f, 0.f, 0.f};

      for (int k = 0; k < KS; ++k) {
        ring_barrier_n<2 * TB, 2 * TB + 3>(last_ops);
        const int sn = st == 0 ? kRing - 1 : st - 1;
        if (k == 0 && out_rows > 0) {
          copy_out(reinterpret_cast<const uint16_t*>(s_b[sn]));
          out_rows = 0;
          lds_barrier();
        }
        if (more) {
          if (k == 0) {
            request_pairs(nxt, pairs, s_pn);
            after = item_fetch<STREAM>(n, ncols, wide, wmax);
          } else if (k == 1) {
            put_rows(nxt, s_pn, 1, npairs, s_pair[nb], s_row[nb]);
          } else if (k == 2) {
            ao_nxt = a_offsets(s_row[nb], I, KB);
            request_scales(nxt, s_row[nb], s_sw[nb], s_w[nb]);
          }
        }
        const int blk = k + kAhead;
        if (blk < KS || !more)
          last_ops = issue(sn, wb_cur, ao_cur, blk < KB ? blk : KB - 1, nmi);
        else
          last_ops = issue(sn, wb_nxt, ao_nxt, blk - KS < KB ? blk - KS : KB - 1, nmi_nxt);
        if (k < KB) {
          const float w = s_sw[cb][(TB * wave / 8) * KB + k];
          u32x4 b[TB][2];
#pragma unroll
          for (int t = 0; t < TB; ++t) read_frag(s_b[st], 16 * TB * wave + 16 * t + j, q, b[t]);
          u32x4 a[2][2];
          float sa[2];
          auto fetch = [&](int mi, int slot) {
            read_frag(s_a[st], 16 * mi + j, q, a[slot]);
            sa[slot] = s_s[st][16 * mi + j];
          };
          fetch(0, 0);
#pragma unroll
          for (int mi = 0; mi < MI; ++mi) {
            const int c = mi & 1;
            if (mi + 1 < MI) fetch(mi + 1, c ^ 1);
#pragma unroll
            for (int t = 0; t < TB; ++t) {
              const f32x4 part = mfma_k128(b[t], a[c]);
              const float sc = sa[c] * w;
#pragma unroll
              for (int r = 0; r < 4; ++r) acc[mi][t][r] = fmaf(part[r], sc, acc[mi][t][r]);
            }
          }
        }
        st = st == kRing - 1 ? 0 : st + 1;
      }

      // bf16(acc x routed weight), staged 64 rows at a time in the weight
      // stage of the last step (no load targets it before the next item's
      // first step); the last round is written out at that step.
      uint16_t* stg = reinterpret_cast<uint16_t*>(s_b[st == 0 ? kRing - 1 : st - 1]);
      constexpr int kRounds = (MI + kStageRows / 16 - 1) / (kStageRows / 16);
#pragma unroll
      for (int rd = 0; rd < kRounds; ++rd) {
        const int r0 = rd * kStageRows;
        if (rd > 0) {  // an earlier round: written out now
          lds_barrier();
          copy_out(stg);
        }
        lds_barrier();  // every wave is done with the last stage, or with the previous round
#pragma unroll
        for (int mi = rd * (kStageRows / 16); mi < MI && mi < (rd + 1) * (kStageRows / 16); ++mi) {
          // A lane's four columns are half of a 16-byte piece of its row;
          // the pieces are rotated by the row's low 4 bits, so that the 16
          // rows of a store spread over the banks.
          const int row = 16 * mi + j;
          const float wgt = s_w[cb][row];
#pragma unroll
          for (int t = 0; t < TB; ++t) {
            const int piece = (2 * (TB * wave + t) + (q >> 1)) ^ j;
            const uint32_t lo = bf16_bits(acc[mi][t][0] * wgt) | (bf16_bits(acc[mi][t][1] * wgt) << 16);
            const uint32_t hi = bf16_bits(acc[mi][t][2] * wgt) | (bf16_bits(acc[mi][t][3] * wgt) << 16);
            *reinterpret_cast<uint2*>(stg + (row - r0) * NC + piece * 8 + (q & 1) * 4) = make_uint2(lo, hi);
          }
        }
        out_cb = cb;
        out_n0 = n0;
        out_r0 = r0;
        out_rows = cur.count - r0 < kStageRows ? cur.count - r0 : kStageRows;
      }
    });
    if (!more) break;
    cur = nxt;
    nxt = after;
    ++n;
    cb = nb;
    ao_cur = ao_nxt;
  }
  lds_barrier();
  copy_out(reinterpret_cast<const uint16_t*>(s_b[st == 0 ? kRing - 1 : st - 1]));
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// out[t] = bf16(sum over k of contrib[t*topk + k]) in fp32, k ascending,
// over the pairs whose id is a valid expert and, given a map, whose expert
// has a slot (the contribution of one without was never written).
template <typename Id>
__global__ void __launch_bounds__(256) topk_sum_kernel(const uint16_t* __restrict__ contrib, int64_t H, int topk,
                                                       const Id* __restrict__ ids, int E,
                                                       const int32_t* __restrict__ expert_map, int slots,
                                                       uint16_t* __restrict__ out) {
  const int64_t t = blockIdx.y;
  const int64_t c = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * 8;
  if (c >= H) return;
  float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  // Eight pairs at a time: the ids and the contribution rows are loaded
  // together (a row is read whatever its id, and skipped in the sum), so
  // the loads do not wait on one another.
  for (int k0 = 0; k0 < topk; k0 += 8) {
    bool ok[8];
    u32x4 v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int k = k0 + i < topk ? k0 + i : topk - 1;
      const int64_t p = t * topk + k;
      const int64_t e = ids[p];
      ok[i] = k0 + i < topk && e >= 0 && e < E;
      if (expert_map && ok[i]) {
        const int sl = expert_map[e];
        ok[i] = sl >= 0 && sl < slots;
      }
      v[i] = *reinterpret_cast<const u32x4*>(contrib + p * H + c);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (!ok[i]) continue;
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        s[2 * w] += bf16_value(v[i][w] & 0xffffu);
        s[2 * w + 1] += bf16_value(v[i][w] >> 16);
      }
    }
  }
  u32x4 o;
#pragma unroll
  for (int i = 0; i < 4; ++i) o[i] = bf16_bits(s[2 * i]) | (bf16_bits(s[2 * i + 1]) << 16);
  *reinterpret_cast<u32x4*>(out + t * H + c) = o;
}

// Routing of npairs pairs, with the quantisation of T tokens where x is given.
int launch_route(const uint16_t* x, int64_t T, int64_t H, uint8_t* xq, float* xs, const void* ids, int eb,
                 int64_t npairs, const int32_t* expert_map, int64_t num_experts, int64_t slots, int32_t* offsets,
                 int32_t* pairs, int32_t* tiles, void* stream) {
  const hipStream_t st = as_stream(stream);
  const int E = static_cast<int>(num_experts), S = static_cast<int>(slots);
  int32_t* wide = npairs > 0 ? tiles + wide_list_offset(npairs, slots) : nullptr;
  const int64_t quant_blocks = x ? (T + 3) / 4 : 0;
  const int nb = route_blocks(npairs);
  if (nb > 0) {
    int32_t* hist = tiles + route_hist_offset(npairs, slots);
    hipLaunchKernelGGL(quant_count_kernel, dim3(static_cast<unsigned>(nb + quant_blocks)), dim3(kRouteThreads), 0, st,
                       x, x ? T : 0, H, xq, xs, ids, eb, npairs, nb, expert_map, E, S, hist);
    if (int rc = check_launch("quant_count_kernel")) return rc;
    hipLaunchKernelGGL(route_scatter_kernel, dim3(static_cast<unsigned>(nb)), dim3(kRouteThreads), 0, st, ids, eb,
                       npairs, expert_map, E, S, hist, offsets, pairs, tiles, wide);
    return check_launch("route_scatter_kernel");
  }
  const size_t lds = static_cast<size_t>(kRouteThreads / 64) * static_cast<size_t>(slots) * sizeof(int);
  if (x) {
    hipLaunchKernelGGL(quant_route_kernel, dim3(static_cast<unsigned>(1 + quant_blocks)), dim3(kRouteThreads), lds,
                       st, x, T, H, xq, xs, ids, eb, npairs, expert_map, E, S, offsets, pairs, tiles, wide);
    return check_launch("quant_route_kernel");
  }
  hipLaunchKernelGGL(route_kernel, dim3(1), dim3(kRouteThreads), lds, st, ids, eb, npairs, expert_map, E, S, offsets,
                     pairs, tiles, wide);
  return check_launch("route_kernel");
}

}  // namespace
}  // namespace xp

using namespace xp;

extern "C" {

int64_t xp_moe_max_tiles(int64_t npairs, int64_t slots) {
  if (npairs <= 0 || slots <= 0) return 0;
  // The tile list, then the wide-tile list (1 + 3 * wide_bound ints) and the
  // routing workgroups' counts, in two-int entries past tiles[0].
  const int64_t ints = route_hist_offset(npairs, slots) - 1 + route_blocks(npairs) * slots;
  return (ints + 1) / 2;
}

int xp_quant_tokens(const uint16_t* x, int64_t T, int64_t H, uint8_t* xq, float* xs, void* stream) {
  XP_REQUIRE(T >= 0 && T <= INT32_MAX && H > 0 && H % kKB == 0,
             "xp_quant_tokens: T=%lld, H=%lld (H must be a positive multiple of %d)", (long long)T, (long long)H,
             kKB);
  if (T == 0) return XP_OK;
  XP_REQUIRE(x && xq && xs && aligned16(x) && aligned16(xq), "xp_quant_tokens: null or misaligned buffer");
  hipLaunchKernelGGL(quant_tokens_kernel, dim3(static_cast<unsigned>(T)), dim3(256), 0, as_stream(stream), x, H, xq,
                     xs);
  return check_launch("quant_tokens_kernel");
}

int xp_moe_route(const void* topk_ids, int topk_elem_bytes, int64_t T, int64_t topk, const int32_t* expert_map,
                 int64_t num_experts, int64_t slots, int32_t* offsets, int32_t* pairs, int32_t* tiles, void* stream) {
  XP_REQUIRE(topk_elem_bytes == 4 || topk_elem_bytes == 8, "xp_moe_route: id size %d", topk_elem_bytes);
  XP_REQUIRE(T >= 0 && topk >= 1 && T * topk <= INT32_MAX, "xp_moe_route: T=%lld, topk=%lld", (long long)T,
             (long long)topk);
  XP_REQUIRE(slots >= 1 && slots <= kMaxRouteSlots, "xp_moe_route: %lld slots (at most %d)", (long long)slots,
             kMaxRouteSlots);
  XP_REQUIRE(num_experts >= 1 && num_experts <= INT32_MAX, "xp_moe_route: %lld experts", (long long)num_experts);
  XP_REQUIRE(expert_map && offsets && pairs && tiles && (T == 0 || topk_ids), "xp_moe_route: null argument");
  return launch_route(nullptr, 0, 0, nullptr, nullptr, topk_ids, topk_elem_bytes, T * topk, expert_map, num_experts,
                      slots, offsets, pairs, tiles, stream);
}

int xp_moe_quant_route(const uint16_t* x, int64_t T, int64_t H, uint8_t* xq, float* xs, const void* topk_ids,
                       int topk_elem_bytes, int64_t topk, const int32_t* expert_map, int64_t num_experts,
                       int64_t slots, int32_t* offsets, int32_t* pairs, int32_t* tiles, void* stream) {
  XP_REQUIRE(T >= 0 && T <= INT32_MAX && H > 0 && H % kKB == 0,
             "xp_moe_quant_route: T=%lld, H=%lld (H must be a positive multiple of %d)", (long long)T,
             (long long)H, kKB);
  XP_REQUIRE(topk_elem_bytes == 4 || topk_elem_bytes == 8, "xp_moe_quant_route: id size %d", topk_elem_bytes);
  XP_REQUIRE(topk >= 1 && T * topk <= INT32_MAX, "xp_moe_quant_route: topk=%lld", (long long)topk);
  XP_REQUIRE(slots >= 1 && slots <= kMaxRouteSlots, "xp_moe_quant_route: %lld slots (at most %d)",
             (long long)slots, kMaxRouteSlots);
  XP_REQUIRE(num_experts >= 1 && num_experts <= INT32_MAX, "xp_moe_quant_route: %lld experts",
             (long long)num_experts);
  XP_REQUIRE(expert_map && offsets && pairs && tiles, "xp_moe_quant_route: null argument");
  XP_REQUIRE(T == 0 || (x && xq && xs && topk_ids && aligned16(x) && aligned16(xq)),
             "xp_moe_quant_route: null or misaligned buffer");
  return launch_route(x, T, H, xq, xs, topk_ids, topk_elem_bytes, T * topk, expert_map, num_experts, slots, offsets,
                      pairs, tiles, stream);
}

int64_t xp_moe_workspace_bytes(int64_t npairs, int64_t I) {
  if (npairs <= 0 || I <= 0) return 0;
  return work_layout(npairs, I, nullptr, nullptr);
}

}  // extern "C"

namespace xp {
namespace {

// Argument checks shared by the expert entry points (all but the
// workspace's and the token operands').
int check_ffn(const char* what, int64_t T, int64_t topk, const float* topk_weight, int64_t H, int64_t I,
              const uint8_t* w13, const float* w13_scale, const uint8_t* w2, const float* w2_scale, int64_t slots,
              const int32_t* offsets, const int32_t* pairs, const int32_t* tiles, const uint16_t* out) {
  XP_REQUIRE(H > 0 && I > 0 && H % kBN == 0 && I % kBN == 0 && H <= kKB * kMaxKB && I <= kKB * kMaxKB,
             "%s: H=%lld and I=%lld must be multiples of %d, at most %d", what, (long long)H, (long long)I, kBN,
             kKB * kMaxKB);
  XP_REQUIRE(T >= 0 && topk >= 1 && T * topk <= INT32_MAX && slots >= 1 && slots <= kMaxRouteSlots,
             "%s: T=%lld, topk=%lld, slots=%lld", what, (long long)T, (long long)topk, (long long)slots);
  if (T == 0) return XP_OK;
  XP_REQUIRE(topk_weight && w13 && w13_scale && w2 && w2_scale && offsets && pairs && tiles && out,
             "%s: null argument", what);
  XP_REQUIRE(aligned16(w13) && aligned16(w2) && aligned16(out), "%s: fp8 and output buffers must be 16-byte aligned",
             what);
  const int64_t bound = tile_bound(T * topk, slots);
  XP_REQUIRE(bound <= 65535, "%s: %lld tiles exceed the launch grid", what, (long long)bound);
  return XP_OK;
}

int check_experts(const char* what, const uint8_t* xq, const float* xs, int64_t T, int64_t topk,
                  const float* topk_weight, int64_t H, int64_t I, const uint8_t* w13, const float* w13_scale,
                  const uint8_t* w2, const float* w2_scale, int64_t slots, const int32_t* offsets,
                  const int32_t* pairs, const int32_t* tiles, const uint16_t* out, int activation) {
  XP_REQUIRE(activation == XP_ACT_SILU || activation == XP_ACT_GELU, "%s: unknown activation %d", what, activation);
  const int rc = check_ffn(what, T, topk, topk_weight, H, I, w13, w13_scale, w2, w2_scale, slots, offsets, pairs,
                           tiles, out);
  if (rc || T == 0) return rc;
  XP_REQUIRE(xq && xs && aligned16(xq), "%s: xq and xs must be non-null, xq 16-byte aligned", what);
  return XP_OK;
}

// Compute units per XCD of the current device (8 XCDs), looked up once per
// device.
int cus_per_xcd(int* out) {
  static std::mutex mu;
  static int cache[64];
  int dev = -1;
  XP_HIP(hipGetDevice(&dev));
  XP_REQUIRE(dev >= 0 && dev < 64, "device %d (at most 64 devices)", dev);
  std::lock_guard<std::mutex> lock(mu);
  if (cache[dev] == 0) {
    int n = 0;
    XP_HIP(hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev));
    cache[dev] = n / 8 > 0 ? n / 8 : 1;
  }
  *out = cache[dev];
  return XP_OK;
}

// The two (or, for few pairs, narrow) GEMM launches of one expert call over a
// workspace of xp_moe_workspace_bytes(T * topk, I) bytes at `work`.
// num_experts: the experts that the T * topk pairs are spread over.
int launch_experts(const uint8_t* xq, const float* xs, int64_t T, int64_t topk, const float* topk_weight, int64_t H,
                   int64_t I, const uint8_t* w13, const float* w13_scale, const uint8_t* w2, const float* w2_scale,
                   int64_t slots, int64_t num_experts, const int32_t* offsets, const int32_t* pairs,
                   const int32_t* tiles, uint8_t* work, uint16_t* out, int act, void* stream) {
  const int64_t npairs = T * topk;
  const int64_t bound = tile_bound(npairs, slots);
  Work w;
  work_layout(npairs, I, &w, work);
  // Prefill-sized calls run persistent workgroups over wide tiles, 128
  // activation (gemm1) or output (gemm2) columns per item, and quantise the
  // activations in gemm1; small calls take 16-row subtiles (more workgroups
  // for few pairs) and the small-batch gemm2 quantises. Every column is
  // computed the same way in both.
  const bool narrow = bound < kWideTiles;
  int rc = XP_OK;
  if (!narrow) {
    XP_REQUIRE(T * H <= UINT32_MAX && npairs * I <= UINT32_MAX,
               "xp_moe_experts: T*H=%lld and T*topk*I=%lld must stay below 2^32 (call over fewer tokens)",
               (long long)(T * H), (long long)(npairs * I));
    int per_xcd = 0;
    rc = cus_per_xcd(&per_xcd);
    if (rc) return rc;
    const int64_t wmax = wide_bound(npairs, slots);
    const int32_t* wide = tiles + wide_list_offset(npairs, slots);
    const int64_t per_xcd_tiles = (wmax + 7) / 8;  // wide tiles of one XCD, at most
    // One workgroup per CU: the operand ring takes most of its LDS.
    const int64_t n1 = std::min<int64_t>(per_xcd, per_xcd_tiles * (I / (16 * kGemmWaves)));
    const bool stream_w = stream_weights(npairs, num_experts);
    auto* gemm1 = act == XP_ACT_GELU
                      ? (stream_w ? gemm1_kernel<XP_ACT_GELU, true> : gemm1_kernel<XP_ACT_GELU, false>)
                      : (stream_w ? gemm1_kernel<XP_ACT_SILU, true> : gemm1_kernel<XP_ACT_SILU, false>);
    hipLaunchKernelGGL(gemm1, dim3(static_cast<unsigned>(8 * n1)), dim3(64 * kGemmWaves), 0, as_stream(stream), xq, xs,
                       H, I, static_cast<int>(topk), w13, w13_scale, pairs, wide, wmax, npairs, w);
    rc = check_launch("gemm1_kernel");
    if (rc) return rc;
    // 256 output columns per item where H allows, else 128.
    const int tb = H % (2 * kBN) == 0 ? 2 : 1;
    const int64_t n2 = std::min<int64_t>(per_xcd, per_xcd_tiles * (H / (tb * kBN)));
    auto* gemm2 = tb == 2 ? (stream_w ? gemm2_kernel<2, true> : gemm2_kernel<2, false>)
                          : (stream_w ? gemm2_kernel<1, true> : gemm2_kernel<1, false>);
    hipLaunchKernelGGL(gemm2, dim3(static_cast<unsigned>(8 * n2)), dim3(64 * kGemmWaves), 0, as_stream(stream), H, I,
                       topk_weight, w2, w2_scale, pairs, wide, wmax, npairs, w, out);
    return check_launch("gemm2_kernel");
  }
  const int64_t tiles8 = (bound + 7) / 8 * 8;  // the XCD-aware grids cover whole groups of 8 tiles
  const int64_t g2 = tiles8 * (H / kBN);
  // 16-row subtiles a tile can have: a tile holds at most min(64, npairs) pairs.
  const int nsub = static_cast<int>(((npairs < kBM ? npairs : kBM) + 15) / 16);
  // Few pairs: 16-row subtiles x 16 columns, the K blocks split over 4 waves.
  const int64_t g1n = tiles8 * nsub * (I / 16);
  XP_REQUIRE(g1n <= INT32_MAX && nsub * g2 <= INT32_MAX, "xp_moe_experts: grid too large");
  if (act == XP_ACT_GELU)
    hipLaunchKernelGGL(gemm1_narrow_kernel<XP_ACT_GELU>, dim3(static_cast<unsigned>(g1n)), dim3(kThreads), 0,
                       as_stream(stream), xq, xs, H, I, static_cast<int>(topk), w13, w13_scale, offsets, pairs, tiles,
                       nsub, w);
  else
    hipLaunchKernelGGL(gemm1_narrow_kernel<XP_ACT_SILU>, dim3(static_cast<unsigned>(g1n)), dim3(kThreads), 0,
                       as_stream(stream), xq, xs, H, I, static_cast<int>(topk), w13, w13_scale, offsets, pairs, tiles,
                       nsub, w);
  rc = check_launch("gemm1_narrow_kernel");
  if (rc) return rc;
  hipLaunchKernelGGL(gemm2_narrow_kernel<kNarrowChunk>, dim3(static_cast<unsigned>(nsub * g2)), dim3(kThreads), 0,
                     as_stream(stream), H, I, topk_weight, w2, w2_scale, offsets, pairs, tiles, nsub, w, out);
  return check_launch("gemm2_narrow_kernel");
}

int launch_topk_sum(const uint16_t* contrib, int64_t T, int64_t topk, int64_t H, const void* ids, int eb,
                    int64_t num_experts, const int32_t* expert_map, int64_t slots, uint16_t* out, void* stream) {
  const dim3 grid(static_cast<unsigned>((H / 8 + 255) / 256), static_cast<unsigned>(T));
  if (eb == 8)
    hipLaunchKernelGGL(topk_sum_kernel<int64_t>, grid, dim3(256), 0, as_stream(stream), contrib, H,
                       static_cast<int>(topk), static_cast<const int64_t*>(ids), static_cast<int>(num_experts),
                       expert_map, static_cast<int>(slots), out);
  else
    hipLaunchKernelGGL(topk_sum_kernel<int32_t>, grid, dim3(256), 0, as_stream(stream), contrib, H,
                       static_cast<int>(topk), static_cast<const int32_t*>(ids), static_cast<int>(num_experts),
                       expert_map, static_cast<int>(slots), out);
  return check_launch("topk_sum_kernel");
}

// Workspace of xp_moe_layer: what the separate calls hand one another, then
// xp_moe_experts' workspace.
struct LayerWork {
  uint8_t* xq;        // [T][H]
  float* xs;          // [T][H/128]
  int32_t* offsets;   // [slots + 1]
  int32_t* pairs;     // [T * topk]
  int32_t* tiles;     // [1 + 2 * max_tiles]
  uint16_t* contrib;  // [T * topk][H]
  uint8_t* ffn;
};

int64_t layer_layout(int64_t T, int64_t topk, int64_t H, int64_t I, int64_t slots, LayerWork* w, uint8_t* base) {
  const int64_t n = T * topk;
  const int64_t sz[7] = {align256(T * H),
                         align256(T * (H / kKB) * 4),
                         align256((slots + 1) * 4),
                         align256(n * 4),
                         align256((1 + 2 * xp_moe_max_tiles(n, slots)) * 4),
                         align256(n * H * 2),
                         work_layout(n, I, nullptr, nullptr)};
  int64_t at[8] = {0};
  for (int i = 0; i < 7; ++i) at[i + 1] = at[i] + sz[i];
  if (w) {
    w->xq = base;
    w->xs = reinterpret_cast<float*>(base + at[1]);
    w->offsets = reinterpret_cast<int32_t*>(base + at[2]);
    w->pairs = reinterpret_cast<int32_t*>(base + at[3]);
    w->tiles = reinterpret_cast<int32_t*>(base + at[4]);
    w->contrib = reinterpret_cast<uint16_t*>(base + at[5]);
    w->ffn = base + at[6];
  }
  return at[7];
}

}  // namespace
}  // namespace xp

extern "C" {

int64_t xp_moe_layer_bytes(int64_t T, int64_t topk, int64_t H, int64_t I, int64_t slots) {
  if (T <= 0 || topk <= 0 || H <= 0 || I <= 0 || slots <= 0) return 0;
  return layer_layout(T, topk, H, I, slots, nullptr, nullptr);
}

int xp_moe_layer(const uint16_t* x, int64_t T, int64_t H, const void* topk_ids, int topk_elem_bytes, int64_t topk,
                 const float* topk_weight, const int32_t* expert_map, int64_t num_experts, int64_t I,
                 const uint8_t* w13, const float* w13_scale, const uint8_t* w2, const float* w2_scale, int64_t slots,
                 void* work, int64_t work_bytes, uint16_t* out, int activation, void* stream) {
  const char* what = "xp_moe_layer";
  XP_REQUIRE(activation == XP_ACT_SILU || activation == XP_ACT_GELU, "%s: unknown activation %d", what, activation);
  XP_REQUIRE(topk_elem_bytes == 4 || topk_elem_bytes == 8, "%s: id size %d", what, topk_elem_bytes);
  XP_REQUIRE(num_experts >= 1 && num_experts <= INT32_MAX, "%s: %lld experts", what, (long long)num_experts);
  XP_REQUIRE(T >= 0 && T <= 65535, "%s: T=%lld (at most 65535)", what, (long long)T);
  XP_REQUIRE(T == 0 || (work && (reinterpret_cast<uintptr_t>(work) & 255) == 0),
             "%s: the workspace must be non-null and 256-byte aligned", what);
  LayerWork w{};
  const int64_t need = xp_moe_layer_bytes(T, topk, H, I, slots);
  if (T > 0) layer_layout(T, topk, H, I, slots, &w, static_cast<uint8_t*>(work));
  int rc = check_ffn(what, T, topk, topk_weight, H, I, w13, w13_scale, w2, w2_scale, slots, w.offsets, w.pairs,
                     w.tiles, out);
  if (rc || T == 0) return rc;
  XP_REQUIRE(work_bytes >= need, "%s: workspace of %lld B, needs %lld", what, (long long)work_bytes, (long long)need);
  XP_REQUIRE(x && topk_ids && aligned16(x), "%s: x and topk_ids must be non-null, x 16-byte aligned", what);
  rc = launch_route(x, T, H, w.xq, w.xs, topk_ids, topk_elem_bytes, T * topk, expert_map, num_experts, slots,
                    w.offsets, w.pairs, w.tiles, stream);
  if (rc) return rc;
  rc = launch_experts(w.xq, w.xs, T, topk, topk_weight, H, I, w13, w13_scale, w2, w2_scale, slots, num_experts,
                      w.offsets, w.pairs, w.tiles, w.ffn, w.contrib, activation, stream);
  if (rc) return rc;
  // Without a map expert e has slot e, so the sum's bound on the ids says it all.
  const int64_t E = expert_map || num_experts < slots ? num_experts : slots;
  return launch_topk_sum(w.contrib, T, topk, H, topk_ids, topk_elem_bytes, E, expert_map, slots, out, stream);
}

int xp_moe_experts_part(const uint8_t* xq, const float* xs, int64_t T, int64_t topk, const float* topk_weight,
                        int64_t H, int64_t I, const uint8_t* w13, const float* w13_scale, const uint8_t* w2,
                        const float* w2_scale, int64_t slots, int64_t num_experts, const int32_t* offsets,
                        const int32_t* pairs, const int32_t* tiles, void* work, int64_t work_bytes, uint16_t* out,
                        int activation, void* stream) {
  int rc = check_experts("xp_moe_experts", xq, xs, T, topk, topk_weight, H, I, w13, w13_scale, w2, w2_scale, slots,
                         offsets, pairs, tiles, out, activation);
  if (rc) return rc;
  XP_REQUIRE(num_experts >= 1 && num_experts <= INT32_MAX, "xp_moe_experts: %lld experts", (long long)num_experts);
  if (T == 0) return XP_OK;
  XP_REQUIRE(work && (reinterpret_cast<uintptr_t>(work) & 255) == 0,
             "xp_moe_experts: the workspace must be non-null and 256-byte aligned");
  const int64_t need = xp_moe_workspace_bytes(T * topk, I);
  XP_REQUIRE(work_bytes >= need, "xp_moe_experts: workspace of %lld B, needs %lld", (long long)work_bytes,
             (long long)need);
  return launch_experts(xq, xs, T, topk, topk_weight, H, I, w13, w13_scale, w2, w2_scale, slots, num_experts, offsets,
                        pairs, tiles, static_cast<uint8_t*>(work), out, activation, stream);
}

int xp_moe_experts(const uint8_t* xq, const float* xs, int64_t T, int64_t topk, const float* topk_weight, int64_t H,
                   int64_t I, const uint8_t* w13, const float* w13_scale, const uint8_t* w2, const float* w2_scale,
                   int64_t slots, const int32_t* offsets, const int32_t* pairs, const int32_t* tiles, void* work,
                   int64_t work_bytes, uint16_t* out, int activation, void* stream) {
  return xp_moe_experts_part(xq, xs, T, topk, topk_weight, H, I, w13, w13_scale, w2, w2_scale, slots, slots, offsets,
                             pairs, tiles, work, work_bytes, out, activation, stream);
}

int xp_moe_experts_noalloc(const uint8_t* xq, const float* xs, int64_t T, int64_t topk, const float* topk_weight,
                           int64_t H, int64_t I, const uint8_t* w13, const float* w13_scale, const uint8_t* w2,
                           const float* w2_scale, int64_t slots, const int32_t* offsets, const int32_t* pairs,
                           const int32_t* tiles, uint16_t* out, int activation, void* stream) {
  int rc = check_experts("xp_moe_experts_noalloc", xq, xs, T, topk, topk_weight, H, I, w13, w13_scale, w2,
                         w2_scale, slots, offsets, pairs, tiles, out, activation);
  if (rc || T == 0) return rc;
  const int64_t need = xp_moe_workspace_bytes(T * topk, I);
  if (need > XP_MOE_SCRATCH_BYTES)
    return fail(XP_E_LIMIT,
                "xp_moe_experts_noalloc: %lld pairs x I=%lld need a workspace of %lld B, above the library's "
                "%lld B; call xp_moe_experts with a workspace instead",
                (long long)(T * topk), (long long)I, (long long)need, (long long)XP_MOE_SCRATCH_BYTES);
  uint8_t* work = nullptr;
  rc = moe_scratch_address(&work);
  if (rc) return rc;
  return launch_experts(xq, xs, T, topk, topk_weight, H, I, w13, w13_scale, w2, w2_scale, slots, slots, offsets,
                        pairs, tiles, work, out, activation, stream);
}

int xp_moe_decode_experts(const uint16_t* x, int64_t T, int64_t H, const void* topk_ids, int topk_elem_bytes,
                          int64_t topk, const float* topk_weight, const int32_t* expert_map,
                          const int32_t* pair_slot, int64_t num_experts, int64_t I, const uint8_t* w13,
                          const float* w13_scale, const uint8_t* w2, const float* w2_scale, int64_t slots, void* work,
                          int64_t work_bytes, uint16_t* out, int activation, void* stream) {
  const char* what = "xp_moe_decode_experts";
  XP_REQUIRE(T >= 0 && topk >= 1 && T * topk <= INT32_MAX, "%s: T=%lld, topk=%lld", what, (long long)T,
             (long long)topk);
  if (T == 0) return XP_OK;
  const int64_t npairs = T * topk;
  if (npairs > kDecodePairs || H > kDecodeMaxH || topk * I > kDecodeActBytes)
    return fail(XP_E_LIMIT,
                "%s: %lld pairs (at most %d), H=%lld (at most %d), topk*I=%lld (at most %d): use the separate calls",
                what, (long long)npairs, kDecodePairs, (long long)H, kDecodeMaxH, (long long)(topk * I),
                kDecodeActBytes);
  XP_REQUIRE(topk_elem_bytes == 4 || topk_elem_bytes == 8, "%s: id size %d", what, topk_elem_bytes);
  XP_REQUIRE(activation == XP_ACT_SILU || activation == XP_ACT_GELU, "%s: unknown activation %d", what, activation);
  XP_REQUIRE(num_experts >= 1 && num_experts <= INT32_MAX, "%s: %lld experts", what, (long long)num_experts);
  XP_REQUIRE(H > 0 && I > 0 && H % kBN == 0 && I % kBN == 0, "%s: H=%lld and I=%lld must be multiples of %d", what,
             (long long)H, (long long)I, kBN);
  XP_REQUIRE(slots >= 1 && slots <= kMaxRouteSlots, "%s: %lld slots (at most %d)", what, (long long)slots,
             kMaxRouteSlots);
  XP_REQUIRE(x && topk_ids && expert_map && topk_weight && w13 && w13_scale && w2 && w2_scale && out,
             "%s: null argument", what);
  XP_REQUIRE(aligned16(x) && aligned16(w13) && aligned16(w2) && aligned16(out), "%s: misaligned buffer", what);
  XP_REQUIRE(work && (reinterpret_cast<uintptr_t>(work) & 255) == 0,
             "%s: the workspace must be non-null and 256-byte aligned", what);
  const int64_t need = xp_moe_workspace_bytes(npairs, I);
  XP_REQUIRE(work_bytes >= need, "%s: workspace of %lld B, needs %lld", what, (long long)work_bytes, (long long)need);
  Work w;
  work_layout(npairs, I, &w, static_cast<uint8_t*>(work));
  // One workgroup per subtile of an occupied slot and 16 columns: 4 or 8 rows
  // where that many tokens cannot fill more of a slot, else 16. With m slots
  // occupied by n pairs, sum over slots of ceil(c / rows) is at most
  // m + (n - m) / rows, which grows with m up to min(n, slots).
  const int rows = T <= 4 ? 4 : T <= 8 ? 8 : 16;
  const int64_t occupied = npairs < slots ? npairs : slots;
  const int64_t subs = occupied + (npairs - occupied) / rows;
  const int64_t subs8 = (subs + 7) / 8 * 8;  // the XCD-aware grid covers whole groups of 8
  const dim3 g1(static_cast<unsigned>(subs8 * (I / 16)));
  const size_t lds = static_cast<size_t>(rows) * static_cast<size_t>(H);
  auto gate_up = [&](auto act_c) {
    constexpr int ACT = decltype(act_c)::value;
    auto* kernel = rows == 4 ? gemm1_decode_kernel<ACT, 4> : rows == 8 ? gemm1_decode_kernel<ACT, 8>
                                                                       : gemm1_decode_kernel<ACT, 16>;
    hipLaunchKernelGGL(kernel, g1, dim3(kThreads), lds, as_stream(stream), x, H, I, topk_ids, topk_elem_bytes,
                       static_cast<int>(npairs), static_cast<int>(topk), expert_map, pair_slot,
                       static_cast<int>(num_experts), static_cast<int>(slots), w13, w13_scale, w);
  };
  if (activation == XP_ACT_GELU)
    gate_up(Int<XP_ACT_GELU>{});
  else
    gate_up(Int<XP_ACT_SILU>{});
  int rc = check_launch("gemm1_decode_kernel");
  if (rc) return rc;
  const int cols = T == 1 ? 8 : 16;
  hipLaunchKernelGGL(cols == 8 ? gemm2_decode_kernel<8> : gemm2_decode_kernel<16>,
                     dim3(static_cast<unsigned>(T * (H / cols))), dim3(kThreads), static_cast<size_t>(topk * I),
                     as_stream(stream), H, I, static_cast<int>(topk), topk_weight, w2, w2_scale, w, out);
  return check_launch("gemm2_decode_kernel");
}

int xp_moe_topk_sum(const uint16_t* contrib, int64_t T, int64_t topk, int64_t H, const void* topk_ids,
                    int topk_elem_bytes, int64_t num_experts, uint16_t* out, void* stream) {
  XP_REQUIRE(T >= 0 && T <= 65535 && topk >= 1 && H > 0 && H % 8 == 0,
             "xp_moe_topk_sum: T=%lld (at most 65535), topk=%lld, H=%lld (a multiple of 8)", (long long)T,
             (long long)topk, (long long)H);
  XP_REQUIRE(topk_elem_bytes == 4 || topk_elem_bytes == 8, "xp_moe_topk_sum: id size %d", topk_elem_bytes);
  if (T == 0) return XP_OK;
  XP_REQUIRE(contrib && out && topk_ids && aligned16(contrib) && aligned16(out),
             "xp_moe_topk_sum: null or misaligned buffer");
  return launch_topk_sum(contrib, T, topk, H, topk_ids, topk_elem_bytes, num_experts, nullptr, 0, out, stream);
}

}  // extern "C"
