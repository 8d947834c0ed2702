"""The low-bit skinny kernel (csrc/hip/lowbit_skinny.cuh) at the edges of its tiles: rows around its 16-row tiles and
64-row blocks, column tails inside a tile and a wave pair, K of half a chunk / an odd number of chunks / more slabs than
chunks, both workgroup sizes, every decoder kind."""
import pytest
import torch

import ipex_llm_amd.ops as ops
from ipex_llm_amd.ops import reference as R
from ipex_llm_amd.quantize import get_format

pytestmark = pytest.mark.gpu


@pytest.fixture
def cuda():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    return torch.device("cuda", 0)


def _rel(a, b):
    a, b = a.double(), b.double()
    return ((a - b).norm() / b.norm()).item()


# 16-bit results: one rounding (2^-9 of a value at most, bf16).  f32 slabs: the offset formats sum codes of up to
# 1032 + 7 in f16 (136 + 7 in bf16) that cancel to a few units, each f32 product sum 2^-24 off: about 1e-5; the table
# formats carry their 16-bit rounded table (2^-9 of a value at most)
STORE, SUM, TABLE = 2 ** -8, 1e-4, 2 ** -8


@pytest.mark.parametrize("name", ["sym_int4", "asym_int4", "nf4", "fp4", "sym_int8", "asym_int5", "fp8_e4m3", "fp8_e5m2"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_rows_and_tails(cuda, name, dtype):
    from ipex_llm_amd.models.decoder import deinterleave_glu
    f = get_format(name).fmt
    torch.manual_seed(1)
    for n, k in [(80, 64), (96, 320), (2080, 640), (4096, 192)]:
        w = torch.randn(n, k, device=cuda) * 0.05
        blob = ops.quantize(w, f)
        W = R.dequantize_device_blob(blob.cpu(), f, n, k).to(cuda).double()
        b = torch.randn(n, device=cuda).to(dtype)
        for M in (17, 32, 33, 64):
            x = torch.randn(M, k, device=cuda).to(dtype)
            ref = x.double() @ W.t()
            y = torch.ops.ipex_llm_amd.gemv(x, blob, f, n, k, b, 0, 0, 0)
            assert y.shape == (M, n) and y.dtype == dtype
            assert _rel(y, ref + b.double()) < STORE, (n, k, M)
            for ks in (0, 1, 3, 7):                     # 7 slabs: more than (80, 64) has chunks
                ws = torch.ops.ipex_llm_amd.gemv(x, blob, f, n, k, None, 1, ks, 0)
                assert ks == 0 or ws.shape[0] == min(ks, -(-k // 128)), (n, k, ks)
                assert _rel(ws.double().sum(0), ref) < (TABLE if name == "nf4" else SUM), (n, k, M, ks)
            if n % 32 == 0:
                g, u = deinterleave_glu(ref)
                for act, fn in ((0, torch.nn.functional.silu),
                                (1, lambda t: torch.nn.functional.gelu(t, approximate="tanh"))):
                    y = torch.ops.ipex_llm_amd.gemv(x, blob, f, n, k, None, 2, 1, act)
                    assert _rel(y, fn(g) * u) < 2 * STORE, (n, k, M, act)


@pytest.mark.parametrize("name", ["sym_int4", "asym_int4", "fp8_e5m2"])
@pytest.mark.parametrize("M", [65, 130, 300, 512])
def test_row_blocks(cuda, name, M):
    """several 64-row blocks: the dispatch of the prefill products takes them, and ops.gemm_rows agrees beyond it"""
    from ipex_llm_amd.models.decoder import deinterleave_glu
    from ipex_llm_amd.ops.gemm import lowbit_gemm, rows_fit
    f = get_format(name).fmt
    torch.manual_seed(2)
    for n, k in [(1312, 704), (192, 2048)]:
        blob = ops.quantize(torch.randn(n, k, device=cuda) * 0.05, f)
        W = R.dequantize_device_blob(blob.cpu(), f, n, k).to(cuda).double()
        x = torch.randn(2, M, k, device=cuda).bfloat16()[1]
        b = torch.randn(n, device=cuda).bfloat16()
        ref = x.double() @ W.t()
        assert rows_fit(M, n, f)
        assert _rel(lowbit_gemm(x, blob, f, n, k, b), ref + b.double()) < STORE
        assert torch.equal(lowbit_gemm(x, blob, f, n, k, b), torch.ops.ipex_llm_amd.gemm_rows(x, blob, f, n, k, b, False, 0))
        g, u = deinterleave_glu(ref)
        y = torch.ops.ipex_llm_amd.gemm_rows(x, blob, f, n, k, None, True, 0)
        assert _rel(y, torch.nn.functional.silu(g) * u) < 2 * STORE


def test_inf_and_nan_rows_stay_in_their_rows(cuda):
    """an infinite / NaN activation reaches its own row only (clamped rows and columns past K add nothing)"""
    f = get_format("sym_int4").fmt
    n, k, M = 96, 192, 20
    torch.manual_seed(3)
    blob = ops.quantize(torch.randn(n, k, device=cuda) * 0.05, f)
    x = torch.randn(M, k, device=cuda).bfloat16()
    clean = torch.ops.ipex_llm_amd.gemv(x, blob, f, n, k, None, 0, 1, 0)
    x[M - 1, 0], x[3, k - 1] = float("inf"), float("nan")
    y = torch.ops.ipex_llm_amd.gemv(x, blob, f, n, k, None, 0, 1, 0)
    rest = [r for r in range(M) if r not in (3, M - 1)]
    assert torch.equal(y[rest], clean[rest]) and not y[3].isfinite().any() and not y[M - 1].isfinite().any()
