"""The split-K epilogue of the 8-phase GEMM (csrc/hip/gemm_8p.hip): 16-byte pieces where the row length allows it, single
elements elsewhere, the same sums either way."""
import pytest
import torch

import ipex_llm_amd.ops as ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 65, 300])
@pytest.mark.parametrize("n", [4, 260, 1020])
@pytest.mark.parametrize("S", [2, 3, 6])
def test_pieces_and_elements_agree(M, n, S):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    ops.require()
    K = 64 * 8
    torch.manual_seed(M + n + S)
    x = torch.randn(M, K, device="cuda").bfloat16()
    w = torch.randn(n + 3, K, device="cuda").bfloat16()
    b = torch.randn(n + 3, device="cuda").bfloat16()
    for f32 in (False, True):
        for extra in (1, 2, 3):                            # rows that are no whole number of 16-byte pieces
            y = torch.ops.ipex_llm_amd.gemm_bf16(x, w[:n], b[:n], f32, 0, False, 0, S)
            z = torch.ops.ipex_llm_amd.gemm_bf16(x, w[:n + extra], b[:n + extra], f32, 0, False, 0, S)
            assert torch.equal(y, z[:, :n])                # the same products, slabs summed in the same order
    ref = x.double() @ w[:n].double().t() + b[:n].double()
    err = (torch.ops.ipex_llm_amd.gemm_bf16(x, w[:n], b[:n], False, 0, False, 0, S).double() - ref).abs()
    assert (err <= 2 ** -8 * ref.abs() + 1e-3).all()       # one bf16 rounding; f32 sums of 512 products of order 1
