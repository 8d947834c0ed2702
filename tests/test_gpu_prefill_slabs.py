"""Split products of many rows that leave their sum to the norm: the bits of the product summed on its own."""
import pytest
import torch

from ipex_llm_amd import ops
from ipex_llm_amd.ops import gemm
from ipex_llm_amd.quantize import get_format

pytestmark = pytest.mark.gpu


# skinny: one slab and several, a row past a block of 64, ragged columns; dense: split by 4 and by 2
@pytest.mark.parametrize("qtype,M,n,k", [("sym_int4", 65, 512, 512), ("sym_int4", 129, 1032, 8192), ("fp8_e5m2", 300, 3584, 18944),
                                         ("nf4", 80, 2048, 4096), ("sym_int4", 513, 1024, 4096), ("nf4", 1024, 4096, 2048)])
def test_norm_of_slabs(cuda, qtype, M, n, k):
    torch.manual_seed(M)
    f = get_format(qtype).fmt
    blob = ops.quantize(torch.randn(n, k, device=cuda) * 0.05, f)
    x = torch.randn(M, k, device=cuda).bfloat16()
    res = torch.randn(M, n, device=cuda).bfloat16()
    w = torch.rand(n, device=cuda).bfloat16() + 0.5
    key = (1 << (M - 1).bit_length(), n, k, False, 0)
    before = gemm._CHOICE.get(key)
    gemm._CHOICE[key] = "g8d"
    try:
        part = gemm.lowbit_slabs(x, blob, f, n, k)
        y = ops.lowbit_matmul(x, blob, f, n, k)
    finally:
        gemm._CHOICE.pop(key)
        if before is not None:
            gemm._CHOICE[key] = before
    assert part.dtype == torch.float32 and part.shape[1:] == (M, n)
    r1, r2 = res.clone(), res.clone()
    o1, _ = ops.add_rms_norm(None, r1, w, 1e-5, partials=part)
    o2, _ = ops.add_rms_norm(y, r2, w, 1e-5)
    assert torch.equal(r1, r2) and torch.equal(o1, o2)


def test_products_that_are_not_split(cuda):
    f = get_format("sym_int4").fmt
    blob = ops.quantize(torch.randn(8192, 256, device=cuda), f)
    x = torch.randn(2048, 256, device=cuda).bfloat16()
    assert gemm.lowbit_slabs(x, blob, f, 8192, 256) is None
    assert gemm.lowbit_slabs(x[:70].requires_grad_(), blob, f, 8192, 256) is None
    with pytest.raises(RuntimeError, match="not split"):
        torch.ops.ipex_llm_amd.gemm_bf16_slabs(x, torch.randn(8192, 256, device=cuda).bfloat16())


@pytest.mark.parametrize("qtype", ["sym_int4", "asym_int4", "nf4", "sym_int8", "fp8_e5m2"])
def test_slabs_of_every_route(cuda, qtype):
    """the number of slabs that shape propagation names is the launch's: decode, one-tile, narrow and skinny kernels"""
    f, o = get_format(qtype).fmt, torch.ops.ipex_llm_amd
    for n, k in [(1040, 2048), (4096, 4096), (512, 256), (8200, 1088), (48, 18944)]:
        blob = ops.quantize(torch.randn(n, k, device=cuda) * 0.05, f)
        for M in (1, 7, 16, 17, 40, 64, 65, 300):
            x = torch.randn(M, k, device=cuda).bfloat16()
            for ks in (0, 3) if M <= 64 else (0,):
                y = o.gemv(x, blob, f, n, k, None, 1, ks, 0) if M <= 64 else o.gemm_rows_slabs(x, blob, f, n, k)
                assert y.shape == (o.gemv_slabs(M, n, k, f, True, ks), M, n)
