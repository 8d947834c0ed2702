"""Measured GEMM dispatch bookkeeping (ops/gemm.py _pick): row buckets and the
cached per-shape choice (the timing itself needs a GPU: tests/test_gpu_kernels.py)."""
import pytest

from ipex_llm_amd.ops import gemm as G


def test_row_buckets():
    assert [G._mbucket(m) for m in (1, 512, 513, 1024, 1025, 8192)] == [1, 512, 1024, 1024, 2048, 8192]


def test_cached_choice_is_shared_within_a_bucket():
    saved = dict(G._CHOICE)
    try:
        G._CHOICE.clear()
        G._CHOICE[(1024, 4096, 4096, False, 0)] = "lib"
        never = lambda: (_ for _ in ()).throw(AssertionError("timed a cached shape"))  # noqa: E731
        assert G._pick((700, 4096, 4096, False, 0), never, never) == "lib"
        assert G._pick((1024, 4096, 4096, False, 0), never, never) == "lib"
        assert G.gemm_choices() == {(1024, 4096, 4096, False, 0): "lib"}
    finally:
        G._CHOICE.clear()
        G._CHOICE.update(saved)


def test_choice_does_not_follow_the_noise_of_a_timing(monkeypatch):
    """two candidates as fast as each other: the same one whichever the clock puts first; a faster one is taken"""
    monkeypatch.setattr(G, "_CHOICE", {})
    monkeypatch.setattr(G, "_AUTOTUNE", True)
    monkeypatch.setattr(G.torch.cuda, "is_current_stream_capturing", lambda: False)

    def pick(*times, key=iter(range(100))):
        monkeypatch.setattr(G, "_time_ms", lambda fns: list(times))
        return G._pick((1024, next(key), 64, False, 0), *[lambda: None] * len(times))
    assert pick(139.1, 140.0) == pick(141.0, 138.9) == "g8d"
    assert pick(82.5, 62.2) == "lib" and pick(1480.4, 1401.9) == "lib" and pick(250.0, 265.0) == "g8d"
    assert pick(100.0, 99.0, 90.0) == "lib1" and pick(100.0, 90.0, 89.0) == "lib"


def test_close_timings_are_settled_by_more_rounds(monkeypatch):
    """rounds as they were read, in which the quickest of three put a pair of 8192 rows on either side of the earlier line and a
    product of 1024 rows on cards of either side of it: the same kernel for each; what is not close is not timed again"""
    monkeypatch.setattr(G, "_CHOICE", {})
    monkeypatch.setattr(G, "_AUTOTUNE", True)
    monkeypatch.setattr(G.torch.cuda, "is_current_stream_capturing", lambda: False)

    def pick(M, first, later, key=iter(range(100))):
        asked = []

        def rounds(fns, n):
            asked.append(n)
            return first if len(asked) == 1 else later
        monkeypatch.setattr(G, "_rounds", rounds)
        return G._pick((M, next(key), 64, True, 0), lambda: None, lambda: None), asked
    steady = [[1500.0, 1437.0], [1506.0, 1443.0], [1510.0, 1440.0], [1498.0, 1434.0], [1503.0, 1439.0], [1501.0, 1442.0]]
    for first in ([[1472.0, 1455.0], [1470.0, 1437.0], [1505.0, 1441.0]], [[1500.0, 1410.0]] * 3, [[1440.0, 1445.0]] * 3):
        assert pick(8192, first, steady) == ("lib", [3, 6])
    for first in ([[134.0, 131.0], [134.4, 136.4], [136.0, 136.3]], [[137.0, 131.0]] * 3, [[134.0, 140.0]] * 3):
        assert pick(1024, first, [[134.5, 132.5]] * 6) == pick(1024, first, [[134.5, 138.0]] * 6) == ("g8d", [3, 6])
    assert pick(1024, [[82.0, 62.0]] * 3, None) == ("lib", [3]) and pick(8192, [[720.0, 620.0]] * 3, None) == ("lib", [3])
    assert pick(2048, [[484.0, 598.0]] * 3, None) == ("g8d", [3])


def test_table_formats_lose_no_bit():
    """nf4 / nf3 weights under bf16 activations: the finer table wherever the fused kernel's f16 one served them, and
    its own gate/up pairs"""
    import torch
    from ipex_llm_amd.quantize import get_format
    bf, hf = torch.bfloat16, torch.float16
    for name in ("nf4", "nf3"):
        f = get_format(name).fmt
        assert not G.rows_take(bf, 96, 28672, 4096, f, glu=True) and not G.rows_take(bf, 64, 4096, 4096, f)
        for M, n, k in ((65, 4096, 4096), (256, 6144, 4096), (128, 12288, 8192)):
            assert G.rows_take(bf, M, n, k, f) and G.rows_fine(bf, M, n, k, f) and not G.rows_fine(hf, M, n, k, f)
        assert G.rows_take(hf, 65, 4096, 4096, f) and G.rows_take(bf, 200, 4096, 4096, f)
        assert G.rows_take(bf, 65, 4096, 14336, f)                # a dense bf16 weight otherwise
        assert not G.rows_fine(bf, 65, 4096, 14336, f) and not G.rows_fine(bf, 200, 4096, 4096, f)
    assert not G.rows_take(bf, 0, 4096, 4096, get_format("sym_int4").fmt)     # no rows: the paths that return nothing
    for name in ("sym_int4", "fp4", "fp8_e5m2", "asym_int5"):
        assert G.rows_take(bf, 65, 4096, 4096, get_format(name).fmt) and not G.rows_fine(bf, 65, 4096, 4096, get_format(name).fmt)


def test_longer_products_keep_the_path_they_had():
    """where the skinny kernel measures longer than the path before it: minima in integer bytes over half a round, pairs
    of many short rounds"""
    import torch
    from ipex_llm_amd.quantize import get_format
    bf = torch.bfloat16

    def take(name, M, n, k, glu=False):
        return G.rows_take(bf, M, n, k, get_format(name).fmt, glu)
    assert not take("asym_int5", 320, 4096, 8192) and take("asym_int5", 256, 4096, 8192) and take("asym_int4", 320, 4096, 8192)
    assert not take("asym_int5", 300, 3584, 3584) and take("asym_int5", 320, 1280, 8192)
    assert not take("fp4", 80, 151936, 1024, True) and take("fp4", 80, 49152, 1024, True) and take("fp4", 80, 57344, 8192, True)
    assert not take("asym_int5", 80, 57344, 8192, True) and take("asym_int5", 80, 37888, 3584, True)


def test_prefetch_asks_what_the_product_asks():
    """a weight is expanded ahead exactly where its product expands it: pairs by the pair's rules"""
    import torch
    import ipex_llm_amd.ops as ops
    from ipex_llm_amd.quantize import get_format
    ops.require()
    bf, f = torch.bfloat16, get_format("sym_int4").fmt
    assert not G.wants_dense(bf, 300, 2048, 4096, f) and not G.wants_dense(bf, 300, 2048, 4096, f, glu=True)
    assert not G.wants_dense(bf, 512, 2048, 4096, f) and G.wants_dense(bf, 512, 2048, 4096, f, glu=True)
    assert not G.wants_dense(bf, 90, 28672, 10240, f, glu=True) and G.wants_dense(bf, 97, 28672, 10240, f, glu=True)
    assert G.wants_dense(bf, 1024, 4096, 4096, f) and not G.wants_dense(bf, 100, 28672, 4096, f, glu=True)


def test_pairs_of_8_bit_floats_up_to_512_rows():
    """gate/up: by the rows alone (a column shard as the whole pair), but for a short K; other formats up to 96 rows"""
    import torch
    from ipex_llm_amd.quantize import get_format
    for dt in (torch.bfloat16, torch.float16):
        for n in (2048, 37888, 151936):
            for name in ("fp8_e4m3", "fp8_e5m2", "fp6"):
                f = get_format(name).fmt
                assert all(G.rows_take(dt, M, n, 3584, f, True) for M in (1, 96, 97, 300, 512))
                assert not G.rows_take(dt, 513, n, 3584, f, True) and not G.rows_take(dt, 97, n, 1024, f, True)
            for name in ("sym_int4", "fp4", "sym_int8", "asym_int4"):
                assert not G.rows_take(dt, 97, n, 3584, get_format(name).fmt, True)


@pytest.mark.parametrize("name", ["sym_int4", "asym_int4", "fp8_e5m2"])
def test_traced_slabs_are_the_plans(name):
    """partial sums under tracing have as many slabs as the launch plan makes, also where that is neither one nor two"""
    import torch
    from torch._subclasses.fake_tensor import FakeTensorMode
    import ipex_llm_amd.ops as ops
    from ipex_llm_amd.quantize import get_format
    ops.require()
    f, o, seen = get_format(name).fmt, torch.ops.ipex_llm_amd, set()
    with FakeTensorMode():
        for M, n, k in [(1, 4096, 4096), (16, 2048, 2048), (20, 1024, 256), (48, 4096, 14336), (300, 3584, 18944), (300, 3584, 3584), (65, 512, 512)]:
            x, blob = torch.empty(M, k, dtype=torch.bfloat16, device="cuda"), torch.empty(64, dtype=torch.uint8, device="cuda")
            S = o.gemv_slabs(M, n, k, f, True)
            seen.add(S)
            assert (o.gemv(x, blob, f, n, k, None, 1, 0, 0) if M <= 64 else o.gemm_rows_slabs(x, blob, f, n, k)).shape == (S, M, n)
            assert o.gemv(x[:1], blob, f, n, k, None, 1, 3, 0).shape[0] == o.gemv_slabs(1, n, k, f, True, 3)
        assert max(seen) > 2
        for M, N, K in [(1024, 4096, 14336), (512, 4096, 4096), (1024, 6144, 4096)]:
            y = o.gemm_bf16_slabs(*(torch.empty(r, K, dtype=torch.bfloat16, device="cuda") for r in (M, N)))
            assert y.shape == (o.gemm_bf16_split(M, N, K), M, N)


def test_a_product_in_one_piece_leaves_no_slabs_to_the_norm():
    """the decoder asks for two slabs at least: of one, f32 and written and read once more, the norm saves nothing"""
    import torch
    from torch._subclasses.fake_tensor import FakeTensorMode
    import ipex_llm_amd.ops as ops
    ops.require()
    with FakeTensorMode():
        blob = torch.empty(64, dtype=torch.uint8, device="cuda")
        for M, n, k, S in [(300, 3584, 3584, 1), (512, 4096, 14336, 1), (300, 3584, 18944, 3), (128, 4096, 4096, 2)]:
            x = torch.empty(M, k, dtype=torch.bfloat16, device="cuda")
            part = G.lowbit_slabs(x, blob, 6 if n == 3584 else 0, n, k, least=2)
            assert (part is None) if S == 1 else part.shape == (S, M, n), (M, n, k)
            assert G.lowbit_slabs(x, blob, 6 if n == 3584 else 0, n, k).shape == (S, M, n)


def test_traced_slabs_of_unknown_rows():
    import torch
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.fx.experimental.symbolic_shapes import ShapeEnv
    import ipex_llm_amd.ops as ops
    ops.require()
    env = ShapeEnv()
    with FakeTensorMode(shape_env=env):
        x = torch.empty(env.create_unbacked_symint(), 64, dtype=torch.bfloat16, device="cuda")
        y = torch.ops.ipex_llm_amd.gemm_rows_slabs(x, torch.empty(64, dtype=torch.uint8, device="cuda"), 0, 96, 64)
        assert isinstance(y.shape[0], torch.SymInt) and y.shape[2] == 96


def test_traced_decode_launches_take_what_the_ops_take():
    """the launches of a decode step that add or scale by parts of the rows' sums, and the step's state, under tracing"""
    import torch
    from torch._subclasses.fake_tensor import FakeTensorMode
    import ipex_llm_amd.ops as ops
    ops.require()
    o, M, H, N = torch.ops.ipex_llm_amd, 3, 256, 512
    with FakeTensorMode():
        new = lambda *s, dtype=torch.bfloat16: torch.empty(s, dtype=dtype, device="cuda")      # noqa: E731
        x, blob, parts = new(M, H), new(64, dtype=torch.uint8), new(M, H // 16, dtype=torch.float32)
        tab, pos, acc = new(64, 64, 2, dtype=torch.float32), new(M, dtype=torch.long), new(M, N, dtype=torch.float32)
        assert o.gemv_accum(x, blob, 0, N, H, acc, 0, None, tab, pos, N, 128, parts, H, 1e-5) is None
        assert o.gemv_accum(x, blob, 0, N, H, acc, 0) is None
        assert o.gemv_rope(x, blob, 0, N, H, None, acc, tab, pos, N, 128, parts, H, 1e-5) is None
        assert o.gemv_row_norm(x, blob, 0, H, H, x, new(M, H), new(H), False, new(M, H), parts) is None
        assert o.gemv_glu_ss(x, blob, 0, N, H, 0, parts, H, 1e-5, True).shape == (M, N // 2)
        bt, lens = new(M, 4, dtype=torch.int32), new(M, dtype=torch.int32)
        assert o.decode_set_state(pos, pos, None, *(new(M, dtype=torch.long) for _ in range(3)), bt, 64,
                                  new(M, dtype=torch.long), lens) is None
