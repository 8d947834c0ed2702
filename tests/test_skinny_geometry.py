"""Launch geometry of the low-bit skinny product (skinny_plan in csrc/torch/ops_hip.cpp): every chunk of K lies in a
slice and every column and row in a workgroup, with as many slabs as asked for, also more than its own search tries."""
import pytest

import ipex_llm_amd.ops as ops
from ipex_llm_amd.quantize import get_format


@pytest.mark.parametrize("M", [17, 33, 64, 65, 300])
@pytest.mark.parametrize("n,k", [(80, 64), (96, 320), (4096, 8320), (4096, 14336), (28672, 4096), (128, 131072)])
@pytest.mark.parametrize("name", ["sym_int4", "asym_int4", "sym_int8"])
def test_covers_the_product(name, M, n, k):
    import torch
    ops.require()
    chunks, f = -(-k // 128), get_format(name).fmt
    for glu, asked in [(True, 0)] + [(False, s) for s in (0, 1, 2, 63, 64, 65, 100, 112, 1000, 10 ** 6)]:
        if glu and n % 32:
            continue
        mt, nw, cpk, blocks, slices = torch.ops.ipex_llm_amd.skinny_geometry(M, n, k, f, glu, asked)
        assert nw in (4, 8) and 2 <= mt <= 4
        assert cpk * slices >= chunks and cpk % 2 == 0
        assert slices == 1 if glu else slices == min(asked, chunks) if asked else 1 <= slices <= 64
        rows = -(-M // (16 * mt))
        assert rows == -(-M // 64) and blocks >= -(-n // (16 * nw)) * rows
        assert nw == 8 or mt < 4 or name == "sym_int4"        # the others' 4-wave kernels of 64 rows spill


@pytest.mark.parametrize("n,k", [(80, 64), (4096, 4096), (6144, 4096), (12288, 8192)])
def test_finer_table(n, k):
    """the kernels it has: three row tiles, or four in 8 waves"""
    import torch
    ops.require()
    for M in (65, 96, 97, 129, 145, 300, 512):
        mt, nw, cpk, _, slices = torch.ops.ipex_llm_amd.skinny_geometry(M, n, k, get_format("nf4").fmt, False, 0, True)
        assert mt == 3 or (mt, nw) == (4, 8)
        assert cpk * slices >= -(-k // 128)


@pytest.mark.parametrize("k", [3584, 4096, 8192])
def test_heads_by_format_and_shape(k):
    """the kernel of an asym_int4 head of 1 to 16 rows does not depend on their number"""
    import torch
    ops.require()
    for n in (32000, 128256, 152064):
        assert all(torch.ops.ipex_llm_amd.skinny_takes(M, n, k, get_format("asym_int4").fmt, False, True) for M in range(1, 17)), n


# every kind of decoder, both sides of the rule's borders; not products whose K v5 cuts by the rows (of 5248 and up, wide outputs)
@pytest.mark.parametrize("name", ["sym_int4", "asym_int4", "fp4", "sym_int8", "asym_int5", "fp8_e4m3", "fp8_e5m2"])
def test_one_kernel_and_split_for_16_rows(name):
    """the kernel and the slabs of a product of 1 to 16 rows do not depend on their number"""
    import torch
    ops.require()
    f, o = get_format(name).fmt, torch.ops.ipex_llm_amd
    for n in (16, 1024, 2048, 2064, 4096, 4112, 4608, 6144, 8192, 8208):
        for k in (64, 1920, 2048, 2176, 3456, 3584, 4096, 4224, 5120):
            if n > 6144 and k > 4096:
                continue
            takes = {o.skinny_takes(M, n, k, f, False, True) for M in range(1, 17)}
            assert len(takes) == 1, (n, k)
            if takes == {True}:
                assert len({tuple(o.skinny_geometry(M, n, k, f, False, 0)) for M in range(1, 17)}) == 1, (n, k)
    for takes, n, k in [(True, 2048, 2048), (False, 6144, 4096), (False, 1024, 1536), (False, 4096, 2048)]:
        assert o.skinny_takes(1, n, k, f, False, True) == takes, (n, k)


# sym_int4 and fp4 pairs of few columns or a long K are slower at one and two rows (the times are beside the rule)
@pytest.mark.parametrize("name,takes,stays", [
    ("sym_int4", [(28672, 4096), (37888, 3584), (16416, 2048), (28672, 8192), (1024, 512)], [(7168, 4096), (14336, 2048), (3584, 8192), (18944, 8192), (28672, 12288)]),
    ("asym_int4", [(28672, 4096), (7168, 4096), (18944, 8192)], [(7168, 8192), (4096, 5120)]),
    ("fp4", [(37888, 2048), (9728, 1024)], [(7168, 4096), (8192, 8192), (28672, 4096)]),
    ("fp8_e5m2", [(37888, 3584), (28672, 4096), (7168, 2048)], [(7168, 4096), (28672, 7168)]),
    ("sym_int8", [(28672, 4096), (7168, 3584)], [(7168, 4096), (7168, 7168)]),
    ("nf4", [], [(28672, 4096), (1024, 512)])])
def test_pairs_by_format_and_shape(name, takes, stays):
    import torch
    ops.require()
    f, o = get_format(name).fmt, torch.ops.ipex_llm_amd
    for want, shapes in ((True, takes), (False, stays)):
        for n, k in shapes:
            assert {o.skinny_takes(M, n, k, f, True, True, 1) for M in range(1, 17)} == {want}, (n, k)


@pytest.mark.parametrize("name", ["sym_int4", "fp4", "nf4", "fp8_e5m2"])
def test_resident_groups(name):
    """four row tiles take 98 KB of LDS: one workgroup per CU, so more than 256 of 4 waves are rounds"""
    import torch
    ops.require()
    geometry, f = torch.ops.ipex_llm_amd.skinny_geometry, get_format(name).fmt
    for M, n, k, glu in [(49, 37888, 3584, True), (64, 37888, 3584, True), (128, 37888, 3584, True), (49, 4608, 3584, False),
                         (64, 4608, 3584, False), (512, 6144, 4096, False), (300, 8192, 1024, False), (256, 10240, 8192, False)]:
        mt, nw = geometry(M, n, k, f, glu, 0)[:2]
        assert (mt, nw) == (4, 8), (M, n, k)
    assert geometry(256, 4096, 4096, f, False, 0)[:2] == [4, 4] and geometry(192, 4608, 3584, f, False, 0)[:2] == [4, 4]
    assert geometry(48, 6144, 4096, f, False, 0)[0] == 3                     # (three row tiles: two 4-wave groups fit)
