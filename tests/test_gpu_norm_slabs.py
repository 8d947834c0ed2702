"""RMSNorm behind a residual add: x and one to nine slabs, rows of one and two vectors a thread (of which not every thread has
one) and of more, against float64, and bit for bit the form that takes every argument (slabs that are cleared behind it)."""
import pytest
import torch

import ipex_llm_amd.ops as ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H", [8, 2048, 3584, 4096, 4104, 5120, 8192, 16384])
@pytest.mark.parametrize("ks", [0, 1, 2, 3, 4, 5, 6, 7, 8, 9])
def test_residual_add_and_norm(cuda, dtype, H, ks):
    torch.manual_seed(H + ks)
    for M in (1, 45):
        part = torch.randn(max(ks, 1), M, H, device=cuda)
        x = part[0].to(dtype) if ks == 0 else None
        res, w = torch.randn(M, H, device=cuda).to(dtype), torch.randn(H, device=cuda).to(dtype)
        r1 = res.clone()
        y, _ = ops.add_rms_norm(x, r1, w, 1e-5, partials=part.clone() if ks else None)
        if ks:
            # the slabs' sum is f32, in their order
            s = part[0].clone()
            for i in range(1, ks):
                s += part[i]
            x = s.to(dtype)
            p2, r2 = part.clone(), res.clone()
            y2, _ = ops.add_rms_norm(None, r2, w, 1e-5, partials=p2, zero_partials=True)
            assert torch.equal(y, y2) and torch.equal(r1, r2) and int((p2[0] != 0).sum()) == 0
        assert torch.equal(r1, (x.float() + res.float()).to(dtype))
        h = r1.double()
        ref = h * torch.rsqrt(h.pow(2).mean(-1, keepdim=True) + 1e-5) * w.double()
        # the normalised value and the product with w are rounded by at most u each (subnormals: half the smallest step);
        # 5 % on top for the f32 sum and root
        u, tiny = torch.finfo(dtype).eps / 2, torch.finfo(dtype).smallest_normal * torch.finfo(dtype).eps
        assert ((y.double() - ref).abs() <= 2.1 * u * ref.abs() + tiny * (1 + w.double().abs())).all()
