"""Training attention: the order of its workgroups (odd numbers of blocks, resident and larger grids, groups of
heads) and scales on both sides of the early factor (train_attn.hip), vs float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
U = 2.0 ** -8                # bf16 holds 8 significant bits: one rounding


def _ref(q, k, v, do, scale, causal):
    """per query head: out, p, dS and what bounds their errors"""
    G, T = q.shape[1] // k.shape[1], q.shape[2]
    k, v = (t.double().repeat_interleave(G, 1) for t in (k, v))
    q, do = q.double(), do.double().transpose(1, 2)
    s = q @ k.transpose(-1, -2) * scale
    if causal:
        s = s.masked_fill(torch.ones(T, T, dtype=torch.bool, device=q.device).triu(1), float("-inf"))
    p = s.softmax(-1)
    out, mag = p @ v, p @ v.abs()
    ds = p * (do @ v.transpose(-1, -2) - (do * out).sum(-1, keepdim=True))
    # dS itself is rounded; the row's delta comes from the rounded result, whose error is 2 U mag
    eds = U * ds.abs() + p * (do.abs() * 2 * U * mag).sum(-1, keepdim=True)
    return q, k, do, p, out, mag, ds, eds


def _near(got, ref, tol):
    assert ((got.double() - ref).abs() <= 1.02 * tol + 1e-6).all()     # 2 %: the f32 scores, exponentials and sums


# 1 block; 5 blocks of a small grid; 8 blocks, 512 and 2048 workgroups; 7 blocks of 7 heads a group; the plain order
@pytest.mark.parametrize("B,T,Hq,Hkv,D,causal", [(1, 64, 4, 2, 128, True), (2, 320, 6, 3, 64, True), (2, 512, 32, 8, 128, True),
                                                 (8, 512, 32, 8, 64, True), (1, 448, 7, 1, 128, True), (3, 192, 4, 4, 128, False)])
def test_blocks(cuda, B, T, Hq, Hkv, D, causal):
    torch.manual_seed(T + Hq)
    q, do = torch.randn(B, Hq, T, D, device=cuda).bfloat16(), torch.randn(B, T, Hq, D, device=cuda).bfloat16()
    k, v = (torch.randn(B, Hkv, T, D, device=cuda).bfloat16() for _ in range(2))
    scale, G = D ** -0.5, Hq // Hkv
    out, lse = torch.ops.ipex_llm_amd.train_attn_fwd(q, k, v, scale, causal)
    dq, dk, dv = torch.ops.ipex_llm_amd.train_attn_bwd(q, k, v, out, lse, do, scale, causal)
    for b in range(B):
        x = slice(b, b + 1)
        Q, K, DO, p, ref, mag, ds, eds = _ref(q[x], k[x], v[x], do[x], scale, causal)
        _near(out[x].transpose(1, 2), ref, 2 * U * mag)

        def group(t):
            return t.view(1, Hkv, G, T, D).sum(2)
        _near(dq[x], scale * ds @ K, scale * (eds @ K.abs() + U * (ds @ K).abs()))
        dvr, dkr = group(p.transpose(-1, -2) @ DO), group(scale * ds.transpose(-1, -2) @ Q)
        _near(dv[x], dvr, group(U * (p.transpose(-1, -2) @ DO.abs())) + U * dvr.abs())
        _near(dk[x], dkr, group(scale * eds.transpose(-1, -2) @ Q.abs()) + U * dkr.abs())


@pytest.mark.parametrize("scale", [0.0, -0.05, 1e-39, 0.5])
@pytest.mark.parametrize("T", [64, 100])
def test_forward_scales(cuda, scale, T):
    torch.manual_seed(T)
    q, k, v = (torch.randn(2, 4, T, 128, device=cuda).bfloat16() for _ in range(3))
    out, _ = torch.ops.ipex_llm_amd.train_attn_fwd(q, k, v, scale, True)
    _, _, _, _, ref, mag, _, _ = _ref(q, k, v, q.transpose(1, 2), scale, True)
    _near(out.transpose(1, 2), ref, 2 * U * mag)
