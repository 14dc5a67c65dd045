"""Which kernels an expert FFN call takes, by sizes alone (CPU, no kernel is launched)."""

import math
import os
import shutil
import subprocess

import pytest
import torch

from vllm_expert_pager import moe

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vllm-expert-pager_amd", "csrc")


# (T, topk, H, I): steps in which the fused launches were measured to be faster
# than the separate calls, and steps in which they were not.
@pytest.mark.parametrize("T, topk, H, I, pays", [
    (1, 8, 2048, 512, True), (5, 8, 2048, 512, True), (6, 8, 2048, 512, False),  # 40 pairs
    (8, 2, 2048, 512, True), (9, 2, 2048, 512, True), (8, 2, 4096, 1024, True), (9, 2, 4096, 1024, False),
    (9, 1, 512, 128, True), (40, 1, 512, 128, True), (41, 1, 512, 128, False), (20, 2, 1024, 256, True),
    (24, 1, 2048, 512, True), (25, 1, 2048, 512, False), (10, 4, 2048, 512, True), (12, 1, 2048, 1024, True),
    (13, 1, 2048, 1024, False), (24, 1, 2688, 384, True), (25, 1, 2688, 384, False), (9, 1, 2816, 128, False),
    (32, 1, 2048, 128, True), (33, 1, 2048, 128, False), (9, 1, 2048, 32768, False), (1, 1, 2048, 32896, False),
    (8, 1, 4224, 128, False),
])
def test_decode_pays(T, topk, H, I, pays):
    x = torch.empty((T, H), dtype=torch.bfloat16)
    ids = torch.empty((T, topk), dtype=torch.int64)
    assert moe.decode_pays(x, ids, I) == pays
    if pays:
        assert moe.decode_fits(x, ids, I)


@pytest.fixture(scope="module")
def tile_split(tmp_path_factory):
    """shares(live, halves): the list indices that each of the 8 XCDs takes, as csrc/tile_split.h has it."""
    if shutil.which("g++") is None:
        pytest.skip("no g++")
    d = tmp_path_factory.mktemp("split")
    src, exe = d / "split.cpp", d / "split"
    src.write_text("""#include <cstdio>
#include "tile_split.h"
int main() {
  for (int live = 0; live <= 400; ++live)
    for (int halves = 0; halves < 2; ++halves)
      for (int x = 0; x < 8; ++x) {
        std::printf("%d %d", live, halves);
        for (int t = 0; t <= live / 8 + 2; ++t) std::printf(" %d", xp::xcd_tile(live, x, t, halves));
        std::printf("\\n");
      }
}
""")
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    shares = {}
    for line in subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.splitlines():
        live, halves, *tiles = map(int, line.split())
        n = sum(w < live for w in tiles)
        # workgroups stop at the first tile that is not there
        assert all(0 <= w < live for w in tiles[:n]) and min(tiles[n:]) >= live
        shares.setdefault((live, bool(halves)), []).append(tiles[:n])
    return lambda live, halves: shares[live, halves]


def test_tile_split_takes_every_tile_once(tile_split):
    for live in range(401):
        for halves in (False, True):
            shares = tile_split(live, halves)
            assert sorted(sum(shares, [])) == list(range(live))
            # the launch's workgroups are sized for ceil(live / 8) tiles an XCD
            assert {len(s) for s in shares} <= {live // 8, -(-live // 8)}


def test_tile_split_shares_falling_popularity(tile_split):
    """Lists whose tiles get lighter from slot to slot, by e^2 in all (experts of one tile each,
    popular ones first). Halves: an XCD has two sixteenths, places p and 15 - p of 16, so the most
    is cosh(15/16) / cosh(1/16) of the least, 1.26 of the mean and a tile of the last 15 more.
    Eighths of the list give one XCD twice the mean."""
    for live in range(96, 401, 5):
        pairs = [math.exp(-2.0 * i / live) for i in range(live)]
        load = {halves: [sum(pairs[i] for i in s) for s in tile_split(live, halves)] for halves in (False, True)}
        mean = sum(pairs) / 8
        assert max(load[True]) < 1.26 * mean + pairs[live // 16 * 16 - 1]
        assert max(load[False]) > 1.9 * mean


def test_tile_split_keeps_an_experts_tiles_together(tile_split):
    """The tiles of an expert, neighbours in the list, are on one XCD but at 7 borders of eighths."""
    for live in (8, 100, 399):
        owner = {t: x for x, s in enumerate(tile_split(live, False)) for t in s}
        assert sum(owner[t] != owner[t + 1] for t in range(live - 1)) == 7
