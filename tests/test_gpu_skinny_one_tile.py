"""The low-bit skinny kernel's one row tile (csrc/hip/lowbit_skinny.cuh), up to 16 rows: rows at both ends of the tile,
column tails inside a tile, a wave pair and a group, K of half a chunk / an odd number of chunks / several turns of the
weight ring, slabs; the row scale of a deferred norm, the maximum of a head's tile, x that starts anywhere."""
import pytest
import torch

import ipex_llm_amd.ops as ops
from ipex_llm_amd.ops import reference as R
from ipex_llm_amd.quantize import get_format

pytestmark = pytest.mark.gpu
NAMES = ["sym_int4", "asym_int4", "nf4", "fp4", "sym_int8", "asym_int5", "fp8_e4m3", "fp8_e5m2"]
# as in test_gpu_skinny.py: one rounding of a 16-bit result; f32 sums of offset codes; a 16-bit table
STORE, SUM, TABLE = 2 ** -8, 1e-4, 2 ** -8


@pytest.fixture
def cuda():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    return torch.device("cuda", 0)


def _rel(a, b):
    a, b = a.double(), b.double()
    return ((a - b).norm() / b.norm()).item()


@pytest.mark.parametrize("name", NAMES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_rows_and_tails(cuda, name, dtype):
    from ipex_llm_amd.models.decoder import deinterleave_glu
    f = get_format(name).fmt
    torch.manual_seed(1)
    for n, k in [(72, 64), (96, 320), (2080, 1088), (8192, 896), (16416, 1088), (33280, 704)]:
        blob = ops.quantize(torch.randn(n, k, device=cuda) * 0.05, f)
        W = R.dequantize_device_blob(blob, f, n, k).to(cuda).double()
        b = torch.randn(n, device=cuda).to(dtype)
        xs = torch.randn(16, k, device=cuda).to(dtype)
        ones = {}
        for M in (1, 2, 7, 15, 16):
            x, ref = xs[:M], xs[:M].double() @ W.t()
            y = torch.ops.ipex_llm_amd.gemv(x, blob, f, n, k, b, 0, 0, 0)
            assert _rel(y, ref + b.double()) < STORE, (n, k, M)
            for ks in (0, 3):
                ws = torch.ops.ipex_llm_amd.gemv(x, blob, f, n, k, None, 1, ks, 0)
                assert _rel(ws.double().sum(0), ref) < (TABLE if name == "nf4" else SUM), (n, k, M, ks)
            if n % 32 == 0:
                g, u = deinterleave_glu(ref)
                y = torch.ops.ipex_llm_amd.gemv(x, blob, f, n, k, None, 2, 1, 0)
                assert _rel(y, torch.nn.functional.silu(g) * u) < 2 * STORE, (n, k, M)
                assert torch.equal(y[:1], ones.setdefault("glu", y[:1])), (n, k, M)      # no row sees another
                ss = torch.rand(M, device=cuda) * k + 1.0
                inv = torch.rsqrt(ss.double() / k + 1e-5)[:, None]
                y = ops.gemv_glu_ss(x, blob, f, n, k, 1, ss, k, 1e-5)
                want = torch.nn.functional.gelu(g * inv, approximate="tanh") * (u * inv)
                assert _rel(y, want) < 2 * STORE, (n, k, M)


@pytest.mark.parametrize("name,k,takes", [("sym_int4", 8192, True), ("asym_int4", 8192, True), ("fp4", 12288, True),
                                          ("fp8_e5m2", 5120, True), ("fp8_e5m2", 8192, False), ("nf4", 8192, False)])
def test_rows_that_the_decode_kernel_cannot_hold(cuda, name, k, takes):
    """the pair of a deferred norm: taken by the skinny kernel where its rule leaves it to a kernel without the LDS for it"""
    from ipex_llm_amd.models.decoder import deinterleave_glu
    f, n = get_format(name).fmt, 1024
    torch.manual_seed(8)
    blob = ops.quantize(torch.randn(n, k, device=cuda) * 0.05, f)
    W = R.dequantize_device_blob(blob, f, n, k).to(cuda).double()
    for M in (5, 16):
        x, ss = torch.randn(M, k, device=cuda).bfloat16(), torch.rand(M, device=cuda) * k + 1.0
        if M == 16 and not takes:
            with pytest.raises(RuntimeError, match="exceeds LDS"):
                ops.gemv_glu_ss(x, blob, f, n, k, 0, ss, k, 1e-5)
            continue
        g, u = deinterleave_glu(x.double() @ W.t() * torch.rsqrt(ss.double() / k + 1e-5)[:, None])
        assert _rel(ops.gemv_glu_ss(x, blob, f, n, k, 0, ss, k, 1e-5), torch.nn.functional.silu(g) * u) < 2 * STORE, M


@pytest.mark.parametrize("name", ["sym_int4", "sym_int8", "fp8_e5m2"])
def test_split_by_rows(cuda, name):
    """a long K whose x does not fit the decode kernel's LDS at these rows, and one just below"""
    f = get_format(name).fmt
    torch.manual_seed(2)
    for n, k in [(48, 18944), (8200, 4096), (4112, 14336)]:
        blob = ops.quantize(torch.randn(n, k, device=cuda) * 0.05, f)
        W = R.dequantize_device_blob(blob, f, n, k).to(cuda).double()
        for M in (1, 8, 9, 16):
            x = torch.randn(M, k, device=cuda).bfloat16()
            ws = torch.ops.ipex_llm_amd.gemv(x, blob, f, n, k, None, 1, 0, 0)
            assert _rel(ws.double().sum(0), x.double() @ W.t()) < SUM, (n, k, M)


@pytest.mark.parametrize("name", NAMES)
@pytest.mark.parametrize("M", [5, 6, 7, 16])
def test_tile_maxima(cuda, name, M):
    """(maximum, index) of every 16-column tile: ties to the first index, NaN and -inf never"""
    f = get_format(name).fmt
    torch.manual_seed(3)
    n, k = 1000 + 8, 576
    w = torch.randn(n, k, device=cuda) * 0.05
    w[21] = w[27]
    blob = ops.quantize(w, f)
    b = torch.zeros(n, device=cuda, dtype=torch.bfloat16)
    b[40], b[100:112] = float("nan"), float("-inf")
    x = torch.randn(M, k, device=cuda).bfloat16()
    x[M - 1] = w[27].bfloat16() * 4
    logits, parts = torch.ops.ipex_llm_amd.gemv_argmax(x, blob, f, n, k, b)
    assert _rel(logits[:, :40], x.double() @ R.dequantize_device_blob(blob, f, n, k).to(cuda).double().t()[:, :40]) < STORE
    v = torch.full((M, parts.shape[0] * 16), float("-inf"), device=cuda)
    v[:, :n] = torch.where(logits.float().isnan(), float("-inf"), logits.float())
    best, at = v.view(M, -1, 16).max(-1)
    first = (v.view(M, -1, 16) == best[..., None]).float().argmax(-1)
    assert torch.equal(parts[..., 0].t(), best)
    idx, want = parts[..., 1].contiguous().view(torch.int32).t(), first + torch.arange(parts.shape[0], device=cuda) * 16
    on = best > float("-inf")
    assert torch.equal(idx[on], want[on].int()) and (idx[~on] == 0x7FFFFFFF).all()


@pytest.mark.parametrize("at", [1, 2, 4])
def test_x_that_starts_anywhere(cuda, at):
    """x as a view whose first element is not 16-byte aligned"""
    f, n, k = get_format("sym_int4").fmt, 4096, 1088
    torch.manual_seed(4)
    blob = ops.quantize(torch.randn(n, k, device=cuda) * 0.05, f)
    for M in (3, 16, 40, 100):
        flat = torch.randn(M * k + 8, device=cuda).bfloat16()
        x = flat[at:at + M * k].view(M, k)
        for epi, op in ((0, torch.ops.ipex_llm_amd.gemv), (2, torch.ops.ipex_llm_amd.gemv)):
            if M > 64:
                y, want = (torch.ops.ipex_llm_amd.gemm_rows(t, blob, f, n, k, None, epi == 2, 0) for t in (x, x.clone()))
            else:
                y, want = (op(t, blob, f, n, k, None, epi, 1, 0) for t in (x, x.clone()))
            assert torch.equal(y, want), (M, epi)


@pytest.mark.parametrize("name", ["sym_int4", "asym_int4", "sym_int8", "fp8_e5m2"])
@pytest.mark.parametrize("n,k", [(2048, 4096), (1040, 2112), (4096, 5120), (6144, 4096), (8192, 4096), (5120, 5120)])
def test_rows_do_not_see_each_other(cuda, name, n, k):
    """plain products and their slabs, on both sides of the rule"""
    f = get_format(name).fmt
    torch.manual_seed(7)
    blob = ops.quantize(torch.randn(n, k, device=cuda) * 0.05, f)
    x = torch.randn(16, k, device=cuda).bfloat16()
    for epi in (0, 1):
        one = torch.ops.ipex_llm_amd.gemv(x[:1], blob, f, n, k, None, epi, 0, 0)
        for M in (2, 7, 8, 10, 11, 13, 16):
            y = torch.ops.ipex_llm_amd.gemv(x[:M], blob, f, n, k, None, epi, 0, 0)
            assert torch.equal(y[:, :1] if epi else y[:1], one), (epi, M)


@pytest.mark.parametrize("name", ["sym_int4", "asym_int4", "nf4", "fp8_e5m2"])
@pytest.mark.parametrize("n,k", [(32000, 3584), (32016, 4096), (1008, 4096)])
def test_a_heads_rows_do_not_see_each_other(cuda, name, n, k):
    """one kernel for 1 to 16 rows: the logits and tile maxima of a row are the same bits beside any other rows, and
    those of the plain product where the skinny kernel takes the head"""
    f = get_format(name).fmt
    torch.manual_seed(6)
    blob = ops.quantize(torch.randn(n, k, device=cuda) * 0.05, f)
    x = torch.randn(16, k, device=cuda).bfloat16()
    one, parts = torch.ops.ipex_llm_amd.gemv_argmax(x[:1], blob, f, n, k, None)
    assert _rel(one, x[:1].double() @ R.dequantize_device_blob(blob, f, n, k).to(cuda).double().t()) < 2 * STORE
    tiles = torch.nn.functional.pad(one.float(), (0, -n % 16), value=float("-inf")).view(-1, 16)
    assert torch.equal(parts[:, 0, 0], tiles.amax(-1))
    assert torch.equal(parts[:, 0, 1].contiguous().view(torch.int32), torch.arange(tiles.shape[0], device=cuda).int() * 16
                       + (tiles == tiles.amax(-1, keepdim=True)).float().argmax(-1).int())
    for M in (2, 5, 6, 8, 15, 16):
        y, p = torch.ops.ipex_llm_amd.gemv_argmax(x[:M], blob, f, n, k, None)
        assert torch.equal(y[:1], one) and torch.equal(p[:, :1], parts), M
        if torch.ops.ipex_llm_amd.skinny_takes(1, n, k, f, False, True):
            assert torch.equal(torch.ops.ipex_llm_amd.gemv(x[:M], blob, f, n, k, None, 0, 0, 0)[:1], one), M


@pytest.mark.parametrize("name", ["fp8_e4m3", "fp8_e5m2", "fp6"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_pairs_of_8_bit_floats(cuda, name, dtype):
    """gate/up products of 97 to 512 rows: row blocks of every height, both sides of the rule"""
    from ipex_llm_amd.models.decoder import deinterleave_glu
    from ipex_llm_amd.ops.gemm import lowbit_gemm_glu, rows_take
    f = get_format(name).fmt
    torch.manual_seed(5)
    for n, k in [(96, 1088), (4128, 1152), (320, 1024)]:
        blob = ops.quantize(torch.randn(n, k, device=cuda) * 0.05, f)
        W = R.dequantize_device_blob(blob, f, n, k).to(cuda).double()
        for M in (97, 129, 300, 385, 511, 512, 513):
            x = torch.randn(M, k, device=cuda).to(dtype)
            assert rows_take(dtype, M, n, k, f, True) == (M <= 512 and k > 1024)
            g, u = deinterleave_glu(x.double() @ W.t())
            assert _rel(lowbit_gemm_glu(x, blob, f, n, k), torch.nn.functional.silu(g) * u) < 2 * STORE, (n, k, M)
