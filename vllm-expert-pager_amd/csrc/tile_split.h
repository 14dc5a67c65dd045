// How the prefill GEMMs (moe.hip) share the wide-tile list out over the 8 XCDs.
//
// The list is in slot order, so the tiles of one expert are neighbours. Where
// experts have several tiles (unmarked weight rows, see dma16_stream), an XCD
// takes one contiguous eighth, so that an expert's tiles read its weight rows
// into one L2. Where most have one, the work of an eighth depends on how popular
// its experts are: with popularity that falls along the slots, the first XCD has
// the full tiles and the last one those of a pair or two. There the list is cut
// in halves, shared out in eighths forwards in the first and backwards in the
// second, which evens a trend out, and the last tiles (below 16) are dealt
// singly.
//
// Both GEMMs with single tiles in turn (and the kernel before the weights became
// the first MFMA operand), with eighths and with halves, relative to the first:
// 256 experts 2048 x 512 at top-8 whose popularity falls by e^2 over the slots,
// 700 tokens 1, 1.19, 1.02 and 1100 tokens 1, 1.27, 0.98; 64 experts 1024 x 1024
// at top-4, 700 tokens 1, 1.28, 0.90; the worst of 57 such lists 1, 1.15, 1.07.
// With popularity in no order (19 sizes, 8 routings each) halves take 0.997 of
// the time of eighths, runs of 2 tiles in turn 1.010, single tiles 1.01. Runs and
// single tiles also make the first pass over new weights 3% longer at 2048
// tokens: each XCD then goes through the whole slab.
#pragma once

namespace xp {

// List index of XCD `xcd`'s tile t, `live` or more if it has none.
constexpr int xcd_tile(int live, int xcd, int t, bool halves) {
  if (halves) {
    const int run = live >> 4;
    return t < 2 * run ? (t < run ? xcd : 14 - xcd) * run + t : 8 * t + xcd;
  }
  const int each = live >> 3, extra = live & 7;  // the first `extra` XCDs take one tile more
  if (t >= each + (xcd < extra ? 1 : 0)) return live;
  return xcd * each + (xcd < extra ? xcd : extra) + t;
}

}  // namespace xp
