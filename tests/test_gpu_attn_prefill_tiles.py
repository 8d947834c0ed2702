"""Prefill attention over long block tables, odd scales, and rows without keys (attn_prefill.hip), vs float64."""
import pytest
import torch

from ipex_llm_amd import ops

pytestmark = pytest.mark.gpu


def _case(dev, Tq, L, Hq, Hkv, D, bs, kv_fp8=0, seed=0):
    g = torch.Generator(device=dev).manual_seed(seed)
    nb = -(-L // bs)
    k = torch.randn(nb, Hkv, bs, D, generator=g, device=dev)
    v = torch.randn(nb, Hkv, bs, D, generator=g, device=dev)
    q = torch.randn(Tq, Hq, D, generator=g, device=dev).bfloat16()
    if kv_fp8:
        dt = torch.float8_e5m2 if kv_fp8 == 1 else torch.float8_e4m3fn
        k, v = k.to(dt), v.to(dt)
        kc, vc = k.view(torch.uint8), v.view(torch.uint8)
    else:
        kc, vc = k.bfloat16(), v.bfloat16()
        k, v = kc, vc
    perm = torch.randperm(nb, generator=g, device=dev)
    inv = torch.argsort(perm)                                   # logical block j lies at inv[j]
    flat = [t.double()[inv].transpose(1, 2).reshape(nb * bs, Hkv, D)[:L] for t in (k, v)]
    if not kv_fp8 and L % bs:                                   # stale slots
        kc[inv[-1], :, L % bs:] = float("nan")
        vc[inv[-1], :, L % bs:] = float("nan")
    return q, kc.contiguous(), vc.contiguous(), inv.to(torch.int32)[None].contiguous(), flat


def _check(got, q, flat, Tq, L, scale, window=0):
    kk, vv = flat
    G = q.shape[1] // kk.shape[1]
    pos = torch.arange(Tq, device=q.device) + L - Tq
    key = torch.arange(L, device=q.device)
    ok = (key[None] <= pos[:, None]) & ((key[None] > pos[:, None] - window) if window else True)
    for h in range(q.shape[1]):
        s = (q[:, h].double() @ kk[:, h // G].t() * scale).masked_fill(~ok, float("-inf"))
        p = torch.nan_to_num(s.softmax(-1))                     # a row without keys: zeros
        # bf16 holds 8 significant bits: p and the result are each rounded by at most 2^-8 of themselves, and
        # |result| <= sum p |v|, so 2^-7 of that sum; 2 % on top for the f32 scores, exponentials and sums
        ref, tol = p @ vv[:, h // G], 1.02 * 2.0 ** -7 * (p @ vv[:, h // G].abs()) + 1e-30
        assert ((got[:, h].double() - ref).abs() <= tol).all(), h


@pytest.mark.parametrize("Hq,Hkv,D", [(4, 2, 128), (2, 1, 64)])
@pytest.mark.parametrize("Tq,L,bs", [(70, 64 * 64, 64), (70, 64 * 64 + 1, 64), (65, 64 * 130 + 5, 64), (33, 128 * 66 + 64, 128),
                                     (64, 64, 64), (1, 64 * 65, 64)])
def test_block_tables(cuda, Tq, L, bs, Hq, Hkv, D):
    """one, two and three loads of 64 block ids, at their edges; a whole and a partial last tile"""
    q, kc, vc, bt, flat = _case(cuda, Tq, L, Hq, Hkv, D, bs, seed=L)
    sl = torch.tensor([L], dtype=torch.int32, device=cuda)
    _check(ops.attn_prefill(q, kc, vc, bt, sl, Tq, D ** -0.5), q, flat, Tq, L, D ** -0.5)


@pytest.mark.parametrize("window", [1, 64, 500])
@pytest.mark.parametrize("kv_fp8", [0, 1, 2])
def test_window_starts_inside_the_table(cuda, window, kv_fp8):
    Tq, L = 130, 64 * 70 + 9
    q, kc, vc, bt, flat = _case(cuda, Tq, L, 4, 2, 128, 64, kv_fp8, seed=window)
    sl = torch.tensor([L], dtype=torch.int32, device=cuda)
    _check(ops.attn_prefill(q, kc, vc, bt, sl, Tq, 0.09, 0.0, window, kv_fp8), q, flat, Tq, L, 0.09, window)


@pytest.mark.parametrize("scale", [0.0, -0.05, 1e-39, 0.5])
@pytest.mark.parametrize("kv_fp8", [0, 2])
def test_scales(cuda, scale, kv_fp8):
    """a factor that is not positive and normal goes on before the row maximum"""
    Tq, L = 90, 150
    q, kc, vc, bt, flat = _case(cuda, Tq, L, 4, 2, 128, 64, kv_fp8, seed=3)
    sl = torch.tensor([L], dtype=torch.int32, device=cuda)
    _check(ops.attn_prefill(q, kc, vc, bt, sl, Tq, scale, 0.0, 0, kv_fp8), q, flat, Tq, L, scale)


@pytest.mark.parametrize("kv_fp8", [0, 1])
@pytest.mark.parametrize("L", [1, 20, 64])
def test_rows_without_keys(cuda, L, kv_fp8):
    """fewer keys than query rows: the first rows, a whole workgroup of them too, are zero"""
    Tq = 150
    q, kc, vc, bt, flat = _case(cuda, Tq, L, 4, 2, 128, 64, kv_fp8, seed=L)
    sl = torch.tensor([L], dtype=torch.int32, device=cuda)
    got = ops.attn_prefill(q, kc, vc, bt, sl, Tq, 0.1, 0.0, 0, kv_fp8)
    assert (got[:Tq - L] == 0).all()
    _check(got, q, flat, Tq, L, 0.1)
