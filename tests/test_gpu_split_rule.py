"""Launch shapes of the decode products of at most 16 rows (plan5 in csrc/torch/ops_hip.cpp) on both sides of their
rules: one round of 8-wave groups for long K and narrow outputs, whole-K 8-bit GLU groups."""
import pytest
import torch

import ipex_llm_amd.ops as ops
from ipex_llm_amd.ops import reference as R
from ipex_llm_amd.quantize import get_format

pytestmark = pytest.mark.gpu


def _rel(a, b):
    a, b = a.double(), b.double()
    return ((a - b).norm() / b.norm()).item()


def _weight(name, n, k):
    f = get_format(name).fmt
    torch.manual_seed(n + k)
    blob = ops.quantize(torch.randn(n, k, device="cuda") * 0.05, f)
    return f, blob, R.dequantize_device_blob(blob.cpu(), f, n, k).to("cuda").double()


# f32 sums: offset codes cancel in 16-bit products summed in f32 (about 1e-5), a table's codes are rounded to 16 bits
@pytest.mark.parametrize("name,tol", [("sym_int4", 1e-4), ("asym_int4", 1e-4), ("nf4", 2 ** -8), ("sym_int8", 1e-4),
                                      ("fp8_e4m3", 1e-4), ("fp8_e5m2", 1e-4)])
@pytest.mark.parametrize("n,k", [(96, 8064), (80, 8192), (4096, 8192), (4112, 8192), (48, 18944), (1040, 8320)])
def test_long_k(cuda_ok, name, tol, n, k):
    f, blob, W = _weight(name, n, k)
    for M in (1, 3, 5, 12, 16):
        x = torch.randn(M, k, device="cuda").bfloat16()
        ref = x.double() @ W.t()
        acc = torch.zeros(M, n, device="cuda")
        torch.ops.ipex_llm_amd.gemv_accum(x, blob, f, n, k, acc, 0)
        assert _rel(acc, ref) < tol, (n, k, M)
        ws = torch.ops.ipex_llm_amd.gemv(x, blob, f, n, k, None, 1, 0, 0)
        assert _rel(ws.double().sum(0), ref) < tol, (n, k, M)


@pytest.mark.parametrize("name", ["sym_int4", "sym_int8", "fp8_e5m2"])
@pytest.mark.parametrize("pairs", [1024, 1025, 2047, 2048, 2049])
def test_glu_groups(cuda_ok, name, pairs):
    from ipex_llm_amd.models.decoder import deinterleave_glu
    n, k = 32 * pairs, 320
    f, blob, W = _weight(name, n, k)
    for M in (2, 3, 8, 16):
        x = torch.randn(M, k, device="cuda").bfloat16()
        g, u = deinterleave_glu(x.double() @ W.t())
        y = torch.ops.ipex_llm_amd.gemv(x, blob, f, n, k, None, 2, 1, 0)
        assert _rel(y, torch.nn.functional.silu(g) * u) < 2 ** -7, (pairs, M)     # one bf16 rounding of each result


@pytest.fixture
def cuda_ok():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
