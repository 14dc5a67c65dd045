// How the prefill GEMMs (moe.hip) share the wide-tile list out over the 8 XCDs.
//
// The list is in slot order, so the tiles of one expert are neighbours. Where
// experts have several tiles (unmarked weight rows, see dma16_stream), an XCD
// takes one contiguous eighth, so that an expert's tiles read its weight rows
// into one L2. Where most have one, a contiguous eighth is only as much work as
// its experts are popular: with popularity that falls along the slots, the
// first XCD has the full tiles and the last one those of a pair or two. There
// the XCDs take runs of kTileRun tiles in turn, and the last, partial turn in
// eighths again, so that no XCD has a tile more than another has by eighths.
//
// Both GEMMs by single tiles in turn, by eighths and by runs of 2, relative to
// the first: 256 experts 2048 x 512 at top-8 whose popularity falls by e^2 over
// the slots, 700 tokens 1, 1.18, 0.96 and 1100 tokens 1, 1.26, 0.95; 64 experts
// 1024 x 1024 at top-4, 700 tokens 1, 1.28, 0.91 (single tiles with the kernel
// before the weights became the first MFMA operand). With popularity in no
// order (16 sizes, 8 routings each) runs of 2 take 0.7% longer than eighths and
// single tiles 1%; runs of 4 and 8 take as long as runs of 2, but 8 leaves short
// lists uneven (64 experts, 333 tokens, falling popularity: 1.13).
#pragma once

namespace xp {

constexpr int kXcds = 8;
constexpr int kTileRun = 2;

// Whole turns of runs in a list of `live` tiles.
constexpr int tile_turns(int live, bool runs) { return runs ? live / (kXcds * kTileRun) : 0; }

// Tiles of XCD `xcd`.
constexpr int xcd_tiles(int live, int xcd, bool runs) {
  const int turns = tile_turns(live, runs);
  const int rest = live - turns * kXcds * kTileRun;
  return turns * kTileRun + rest / kXcds + (xcd < rest % kXcds ? 1 : 0);
}

// List index of the XCD's tile t (0 <= t < xcd_tiles).
constexpr int xcd_tile(int live, int xcd, int t, bool runs) {
  const int turns = tile_turns(live, runs);
  if (t < turns * kTileRun) return (t / kTileRun * kXcds + xcd) * kTileRun + t % kTileRun;
  const int rest = live - turns * kXcds * kTileRun, extra = rest % kXcds;
  return live - rest + xcd * (rest / kXcds) + (xcd < extra ? xcd : extra) + t - turns * kTileRun;
}

}  // namespace xp
