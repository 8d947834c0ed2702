"""Decode attention, head dim 128: where a workgroup streams a pair's keys, in how many waves and workgroups (v4_plan in
attn_dec_v4.cuh), at the edges of its rule."""
import pytest

import ipex_llm_amd.ops as ops


@pytest.mark.parametrize("batch,heads,keys,plan", [
    (17, 8, 64, [8, 1]), (32, 8, 2560, [8, 1]), (33, 8, 64, [4, 1]), (100, 8, 640, [4, 1]), (33, 8, 1280, [4, 1]),  # one a pair
    # longer grids: 8 tiles in a row a workgroup, more past 32 workgroups a pair or 8192, so that one long sequence is not one's
    (32, 8, 2624, [4, 3]), (33, 8, 1344, [4, 2]), (32, 8, 16000, [4, 16]), (17, 8, 1 << 20, [4, 32]), (32, 8, 1 << 20, [4, 32]),
    (64, 8, 16384, [4, 16]), (64, 8, 32768, [4, 16]), (200, 8, 32768, [4, 8]), (100, 4, 3008, [4, 3]),
    (4, 32, 64, [0, 0]), (4, 32, 128, [0, 0]), (4, 32, 896, [0, 0]), (4, 32, 960, [4, 4]),         # up to 8 sequences, few keys
    (5, 32, 128, [0, 0]), (8, 32, 512, [0, 0]), (8, 32, 576, [8, 1]), (8, 40, 512, [0, 0]), (8, 40, 576, [4, 1]), (9, 32, 64, [4, 1]),
    (1, 8, 64, [0, 0]), (8, 8, 192, [0, 0]), (9, 8, 192, [4, 1]), (9, 8, 256, [8, 1]), (9, 2, 512, [8, 1]), (9, 2, 576, [0, 0]),
    (9, 8, 704, [8, 1]), (8, 8, 768, [0, 0]), (14, 8, 896, [8, 1]), (14, 8, 960, [4, 4]), (16, 8, 1088, [4, 4]),
    (8, 8, 960, [0, 0]), (8, 8, 1024, [4, 8]), (10, 8, 1088, [0, 0]), (10, 8, 1152, [4, 6]),
    (1, 8, 1856, [0, 0]), (1, 8, 1920, [4, 15]), (1, 8, 4096, [4, 16]), (1, 8, 16384, [4, 32]), (2, 8, 16384, [4, 16]),
    (3, 8, 20032, [4, 16]), (5, 8, 4224, [4, 12]), (1, 1, 1 << 20, [4, 32])])
def test_plan(batch, heads, keys, plan):
    import torch
    ops.require()
    assert torch.ops.ipex_llm_amd.attn_decode_plan(batch, heads, keys // 64) == plan
