"""Which kernels an expert FFN call takes, by sizes alone (CPU, no kernel is launched)."""

import pytest
import torch

from vllm_expert_pager import moe


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
