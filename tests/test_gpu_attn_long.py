"""The long-context decode kernel (csrc/hip/attn_dec_v3.cuh, several 32-key tiles per wave) against RoPE + KV append
followed by the one-tile kernel: sequence ends at and around a tile, a wave row, a split; one short sequence beside long
ones; rotation in the kernel (with bias) and before it; windows; the accumulator left zero and the tickets reset."""
import pytest
import torch

import ipex_llm_amd.ops as ops
from ipex_llm_amd.engine.runner import nsplit_for

pytestmark = pytest.mark.gpu


def _rel(a, b):
    a, b = a.double(), b.double()
    return ((a - b).norm() / b.norm()).item()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("prerot", [False, True])
@pytest.mark.parametrize("L", [[3073, 1], [4096, 4097], [5000, 3333], [6144, 6143], [3200, 32, 33, 3105]])
@pytest.mark.parametrize("window", [0, 700])
def test_matches_append_and_one_tile_kernel(dtype, prerot, L, window):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    cuda = torch.device("cuda", 0)
    torch.manual_seed(3)
    D, bs, B, Hq, Hkv = 128, 64, len(L), 32, 8
    nb = (max(L) + bs - 1) // bs
    # >= 48 splits and more than 256 workgroups of one tile per wave: the rule takes the long kernel
    ns = nsplit_for(max(L))
    assert ns >= 48 and B * Hkv * ((ns + 1) // 2) > 256
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
    ref = ops.attn_decode(q.view(B, 1, Hq, D), kc1, vc1, bt, lens, ns, D ** -0.5, window=window)
    for _ in range(3):
        kc2, vc2, p2 = kc.clone(), vc.clone(), part.clone()
        got = ops.attn_decode_rope(p2, bias, cs, pos, kc2, vc2, bt, lens, ns, D ** -0.5, 0.0, window, Hq, D, False, 1.0,
                                   dtype, prerot=prerot)
        assert torch.equal(kc1, kc2) and torch.equal(vc1, vc2)
        # the weights of a key are rounded to 16 bits against another running maximum: 2^-9 (bf16) each at most,
        # averaged over the keys; one rounding of the result
        assert _rel(got, ref) < (2 ** -8 if dtype == torch.bfloat16 else 2 ** -11)
        assert int((p2 != 0).sum()) == 0
    ops.check_kernel_errors(cuda)
