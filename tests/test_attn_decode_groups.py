"""Decode attention of head dim 64: where a wave takes several tiles (v3_long_grid in attn_dec_v3.cuh)."""
import pytest

import ipex_llm_amd.ops as ops


@pytest.mark.parametrize("batch,heads,keys,groups", [
    (31, 8, 4096, 0), (32, 8, 4096, 3), (48, 8, 768, 2), (64, 8, 384, 1), (100, 8, 640, 1),
    (64, 4, 640, 3), (96, 4, 1280, 2), (33, 8, 2560, 2),
    (64, 8, 256, 0), (48, 8, 128, 0),              # one tile a workgroup, or a grid of two
    (32, 8, 512, 0), (32, 8, 576, 3),              # 8-wave groups of one tile per wave: one round, more
    (64, 4, 448, 0), (36, 8, 384, 2),
    (33, 8, 1536, 0), (72, 4, 1280, 0), (41, 8, 1152, 0), (33, 8, 1024, 2), (42, 8, 1536, 2), (33, 8, 1600, 2)])
def test_workgroups_per_pair(batch, heads, keys, groups):
    import torch
    ops.require()
    assert torch.ops.ipex_llm_amd.attn_decode_groups(batch, heads, keys // 64) == groups
