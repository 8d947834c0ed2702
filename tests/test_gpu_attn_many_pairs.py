"""Decode attention of many sequences with q from memory, vs float64; one-token steps and rows of a verify alike.  Head dim
64: several tiles per wave from 256 pairs of sequence and kv head on (attn_dec_v3.cuh, v3_long_grid), one to three workgroups
a pair; head dim 128: streamed (attn_dec_v4.cuh)."""
import pytest
import torch

import ipex_llm_amd.ops as ops
from ipex_llm_amd.engine.runner import nsplit_for

pytestmark = pytest.mark.gpu
EDGES = [1, 31, 32, 33, 64, 127, 128, 129, 255, 256, 257, 383, 384, 385, 500, 700]


def _case(dev, B, Hkv, G, D, dtype, Tq=1, cap=768):
    torch.manual_seed(B * Hkv + D)
    bs, nb = 64, cap // 64
    L = [min(cap, max(EDGES[i % len(EDGES)], Tq)) for i in range(B)]
    kc, vc = (torch.randn(nb * B, Hkv, bs, D, device=dev).to(dtype) for _ in range(2))
    bt = torch.randperm(nb * B, device=dev).int().view(B, nb).contiguous()
    q = torch.randn(B, Tq, Hkv * G, D, device=dev).to(dtype)
    return L, kc, vc, bt, q, torch.tensor(L, dtype=torch.int32, device=dev), nsplit_for(cap)


def _check(got, L, kc, vc, bt, q, scale, softcap, window, alibi):
    B, Tq, Hq, D = q.shape
    Hkv, u = kc.shape[1], torch.finfo(q.dtype).eps / 2
    for b, n in enumerate(L):
        k, v = (c[bt[b].long()].transpose(1, 2).reshape(-1, Hkv, D)[:n].double().repeat_interleave(Hq // Hkv, 1) for c in (kc, vc))
        s = torch.einsum("thd,lhd->htl", q[b].double(), k) * scale
        s = softcap * torch.tanh(s / softcap) if softcap else s
        key, pos = torch.arange(n, device=q.device), torch.arange(Tq, device=q.device)[:, None] + n - Tq
        if alibi is not None:
            s = s + alibi.double()[:, None, None] * key
        ok = (key <= pos) & ((key > pos - window) if window else True)
        p = s.masked_fill(~ok, float("-inf")).softmax(-1)
        ref, mag = torch.einsum("htl,lhd->thd", p, v), torch.einsum("htl,lhd->thd", p, v.abs())
        # p and the result are each rounded by at most u; 5 % on top for the f32 scores, exponentials and sums
        assert ((got[b].double() - ref).abs() <= 2.1 * u * mag + 1e-30).all(), (b, n)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,Hkv,G,D,softcap,window,slopes", [
    (31, 8, 4, 128, 0.0, 0, False),
    (32, 8, 4, 128, 0.0, 0, False),
    (48, 8, 4, 128, 30.0, 0, False),
    (64, 4, 7, 128, 0.0, 100, False),     # groups of 7, a window
    (100, 8, 1, 128, 0.0, 0, False),
    (31, 8, 4, 64, 0.0, 0, False),        # 248 pairs: one tile per wave
    (32, 8, 4, 64, 0.0, 0, False),        # 256: three workgroups a pair
    (48, 8, 4, 64, 30.0, 0, False),       # two
    (64, 4, 7, 64, 0.0, 100, False),      # three, groups of 7, a window
    (130, 4, 8, 64, 0.0, 0, True),        # two, ALiBi
    (100, 8, 1, 64, 0.0, 0, False)])      # 800: one
@pytest.mark.parametrize("cap", [768, 192])   # 6 tiles; 2: one tile per wave
def test_decode(cuda, B, Hkv, G, D, softcap, window, slopes, cap, dtype):
    L, kc, vc, bt, q, sl, ns = _case(cuda, B, Hkv, G, D, dtype, cap=cap)
    alibi = torch.linspace(0.01, 0.5, Hkv * G, device=cuda) if slopes else None
    if D == 64:
        groups = 0 if cap < 256 or B * Hkv < 256 else min(3, max(1, 768 // (B * Hkv)))
        assert torch.ops.ipex_llm_amd.attn_decode_groups(B, Hkv, ns) == groups
    else:
        assert torch.ops.ipex_llm_amd.attn_decode_plan(B, Hkv, ns)[1] == 1
    got = ops.attn_decode(q, kc, vc, bt, sl, ns, D ** -0.5, softcap, window, alibi=alibi)
    _check(got.view_as(q), L, kc, vc, bt, q, D ** -0.5, softcap, window, alibi)
    ops.check_kernel_errors(cuda)


@pytest.mark.parametrize("D", [64, 128])
def test_verify_rows_equal_one_token_steps(cuda, D):
    L, kc, vc, bt, q, sl, ns = _case(cuda, 40, 8, 4, D, torch.bfloat16, Tq=3)
    got = ops.attn_decode(q, kc, vc, bt, sl, ns, 0.1, 0.0, 0).view_as(q)
    _check(got, L, kc, vc, bt, q, 0.1, 0.0, 0, None)
    for t in range(3):
        one = ops.attn_decode(q[:, t:t + 1].contiguous(), kc, vc, bt, sl - (2 - t), ns, 0.1, 0.0, 0)
        assert torch.equal(one.view_as(got[:, t:t + 1]), got[:, t:t + 1])
