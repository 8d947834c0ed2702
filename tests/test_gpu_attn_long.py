"""Decode attention of long contexts over the qkv product's sums against float64: rotation in the kernel (several 32-key
tiles per wave, csrc/hip/attn_dec_v3.cuh) and before it (csrc/hip/attn_dec_v4.cuh).  Sequence ends at and around a tile, a wave
row, a split; short sequences beside long ones and in a grid made for long ones; up to 8 tiles per wave; windows; softcap;
groups of 4 and 7; q, k and v rotated and appended as RoPE + KV append does; the accumulator left zero and the tickets reset."""
import pytest
import torch

import ipex_llm_amd.ops as ops
from ipex_llm_amd.engine.runner import nsplit_for

pytestmark = pytest.mark.gpu


def _rel(a, b):
    a, b = a.double(), b.double()
    return ((a - b).norm() / b.norm()).item()


def _float64(q, kc, vc, bt, n, softcap, window, new=None):
    """q [Hq, D] over the first n keys of a table (the last one replaced by ``new``)"""
    Hkv, D = kc.shape[1], kc.shape[3]
    k, v = (c[bt.long()].transpose(1, 2).reshape(-1, Hkv, D)[:n].double() for c in (kc, vc))
    if new is not None:
        k[-1], v[-1] = new.double()
    s = torch.einsum("hgd,lhd->hgl", q.double().view(Hkv, -1, D), k) * D ** -0.5
    s = softcap * torch.tanh(s / softcap) if softcap else s
    if window:
        s[..., :max(0, n - window)] = float("-inf")
    return torch.einsum("hgl,lhd->hgd", s.softmax(-1), v).reshape(q.shape)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("prerot", [False, True])
@pytest.mark.parametrize("L", [[3585, 1], [4096, 4097], [5000, 3333], [6144, 6143], [4000, 32, 33, 3105]])
@pytest.mark.parametrize("window", [0, 700])
def test_matches_append_and_float64(dtype, prerot, L, window):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    cuda = torch.device("cuda", 0)
    torch.manual_seed(3)
    D, bs, B, Hq, Hkv = 128, 64, len(L), 32, 8
    nb = (max(L) + bs - 1) // bs
    ns = nsplit_for(max(L))
    assert ns >= 56 and torch.ops.ipex_llm_amd.attn_decode_plan(B, Hkv, ns)[1] > 1     # either way in a long kernel
    kc = torch.randn(nb * B, Hkv, bs, D, device=cuda).to(dtype)
    vc = torch.randn(nb * B, Hkv, bs, D, device=cuda).to(dtype)
    bt = torch.randperm(nb * B, device=cuda).int().view(B, nb).contiguous()
    lens = torch.tensor(L, dtype=torch.int32, device=cuda)
    pos = (lens - 1).long()
    W = (Hq + 2 * Hkv) * D
    part = torch.randn(B, W, device=cuda)
    bias = None if prerot else (torch.randn(W, device=cuda) * 0.1).to(dtype)
    fr = torch.arange(max(L), device=cuda).float()[:, None] / (10000 ** (torch.arange(0, D, 2, device=cuda).float() / D))
    cs = torch.stack([fr.cos(), fr.sin()], -1).contiguous()
    if prerot:                      # rotated columns handed over as they are: the oracle rotates by nothing
        cs = torch.stack([torch.ones_like(fr), torch.zeros_like(fr)], -1).contiguous()
    kc1, vc1 = kc.clone(), vc.clone()
    q = torch.empty(B, Hq, D, device=cuda, dtype=dtype)
    ops.rope_kv_fused(part.clone().unsqueeze(0), bias, q, kc1, vc1, pos, bt, 1, cs, Hq, Hkv, D, D, False)
    ref = torch.stack([_float64(q[b], kc1, vc1, bt[b], n, 0.0, window) for b, n in enumerate(L)])
    for _ in range(3):
        kc2, vc2, p2 = kc.clone(), vc.clone(), part.clone()
        got = ops.attn_decode_rope(p2, bias, cs, pos, kc2, vc2, bt, lens, ns, D ** -0.5, 0.0, window, Hq, D, False, 1.0,
                                   dtype, prerot=prerot)
        assert torch.equal(kc1, kc2) and torch.equal(vc1, vc2)
        # probabilities and the result each rounded once
        assert _rel(got.view(B, Hq, D), ref) < torch.finfo(dtype).eps
        assert int((p2 != 0).sum()) == 0
    ops.check_kernel_errors(cuda)


def _tiles(B, Hkv, ns):
    """tiles per wave of a sequence as long as the grid, rotated in the kernel (v3_long_grid)"""
    every = -(-ns * 64 // 128)
    s = min((-(-B * Hkv * -(-every // t) // 256) * (10 * t + 7) + 2 * t, t, -(-every // t)) for t in range(2, 9))[2]
    return -(-every // s)


@pytest.mark.parametrize("prerot", [False, True])
@pytest.mark.parametrize("L,cap,Hkv,G,softcap,window,tiles,plan", [
    ([20000, 10001, 1025], 20000, 8, 4, 0.0, 0, 5, [4, 16]),
    ([6000, 5999, 3001, 129, 64, 4500, 6001, 2, 5000, 4097], 6016, 4, 7, 30.0, 0, 4, [4, 12]),
    ([4096, 4095, 3073, 3072, 1024, 2049, 33, 1], 4096, 32, 1, 0.0, 0, 8, [4, 4]),
    ([4000, 3969, 3968, 1], 4032, 8, 4, 0.0, 1000, 4, [4, 16]),
    ([1000, 64, 1, 129, 130, 3333], 16384, 2, 7, 0.0, 0, 2, [4, 32]),      # a table made for far longer sequences
])
def test_matches_float64(L, cap, Hkv, G, softcap, window, tiles, plan, prerot):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    cuda = torch.device("cuda", 0)
    torch.manual_seed(4)
    D, bs, B, Hq, dtype = 128, 64, len(L), Hkv * G, torch.bfloat16
    nb = -(-cap // bs)
    ns = nsplit_for(cap)
    assert ns >= 48 and _tiles(B, Hkv, ns) == tiles and torch.ops.ipex_llm_amd.attn_decode_plan(B, Hkv, ns) == plan
    kc, vc = (torch.randn(nb * B, Hkv, bs, D, device=cuda).to(dtype) for _ in range(2))
    bt = torch.randperm(nb * B, device=cuda).int().view(B, nb).contiguous()
    lens = torch.tensor(L, dtype=torch.int32, device=cuda)
    part = torch.randn(B, (Hq + 2 * Hkv) * D, device=cuda).to(dtype).float()
    cs = torch.stack([torch.ones(cap, D // 2, device=cuda), torch.zeros(cap, D // 2, device=cuda)], -1).contiguous()
    ref = torch.empty(B, Hq, D, dtype=torch.float64, device=cuda)
    for b, n in enumerate(L):
        ref[b] = _float64(part[b, :Hq * D].view(Hq, D), kc, vc, bt[b], n, softcap, window, part[b, Hq * D:].view(2, Hkv, D))
    for _ in range(2):
        p, k2, v2 = part.clone(), kc.clone(), vc.clone()
        got = ops.attn_decode_rope(p, None, cs, (lens - 1).long(), k2, v2, bt, lens, ns, D ** -0.5, softcap, window, Hq, D,
                                   False, 1.0, dtype, prerot=prerot)        # (the rotation is by nothing)
        # probabilities and the result each rounded once to bf16
        assert _rel(got.view(B, Hq, D), ref) < 2 ** -8
        assert int((p != 0).sum()) == 0
    ops.check_kernel_errors(cuda)


@pytest.mark.parametrize("prerot", [False, True])
def test_values_out_of_the_window_are_not_seen(prerot):
    """infinite and NaN values that left the window (an overflowed f16 cache) change nothing, whole tiles before it"""
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    cuda = torch.device("cuda", 0)
    torch.manual_seed(5)
    D, bs, Hkv, G, L, window = 128, 64, 8, 4, 8192, 700
    B, Hq, nb, ns = 4, Hkv * G, L // bs, nsplit_for(L)
    assert _tiles(B, Hkv, ns) >= 3 and torch.ops.ipex_llm_amd.attn_decode_plan(B, Hkv, ns) == [4, 16]
    kc, vc = (torch.randn(nb * B, Hkv, bs, D, device=cuda).half() for _ in range(2))
    bt = torch.arange(nb * B, device=cuda).int().view(B, nb).contiguous()
    lens = torch.tensor([L, L - 31, L - 400, 3000], dtype=torch.int32, device=cuda)
    part = torch.randn(B, (Hq + 2 * Hkv) * D, device=cuda)
    cs = torch.stack([torch.ones(L, D // 2, device=cuda), torch.zeros(L, D // 2, device=cuda)], -1).contiguous()

    def run(v):
        return ops.attn_decode_rope(part.clone(), None, cs, (lens - 1).long(), kc.clone(), v, bt, lens, ns, D ** -0.5, 0.0,
                                    window, Hq, D, False, 1.0, torch.float16, prerot=prerot)
    clean, bad = run(vc.clone()), vc.clone()
    for b, n in enumerate(lens.tolist()):
        out = (n - window) // 32 * 32                          # the keys before the first tile that holds a visible one
        rows = bad.view(B, nb, Hkv, bs, D)[b].transpose(1, 2).reshape(nb * bs, Hkv, D)
        rows[:out:3], rows[1:out:5] = float("inf"), float("nan")
        bad.view(B, nb, Hkv, bs, D)[b] = rows.view(nb, bs, Hkv, D).transpose(1, 2)
    assert not bad.isfinite().all()
    assert torch.equal(run(bad), clean)
