"""A decode step's qkv projection that stores q as the attention takes it and the new token's k and v in the paged cache: the
values of ``gemv_rope``, rounded once, at the edges of blocks and tables, and nothing anywhere else."""
import pytest
import torch

import ipex_llm_amd.ops as ops
from ipex_llm_amd.quantize import get_format

BS = 64


def _case(q, Hq, Hkv, D, k, M, dtype, dev):
    torch.manual_seed(M * 7 + D)
    n, fmt = (Hq + 2 * Hkv) * D, get_format(q).fmt
    blob = ops.quantize((torch.randn(n, k) * 0.05).to(dev), fmt)
    x = torch.randn(M, k, dtype=dtype)
    tab, pos = torch.randn(512, D // 2, 2), torch.randint(0, 512, (M,))
    # keys on both sides of a block's edge, the last of the table, none (a padding row), one past the table, a bad block
    lens = torch.tensor([1, BS, BS + 1, 3 * BS, 0, 3 * BS + 1, 2 * BS, 70][:M] + [2 * BS + 1 + m for m in range(M - 8)], dtype=torch.int32)
    bt = torch.randperm(3 * M).int().view(M, 3)
    if M > 7:
        bt[7, 1] = 3 * M + 5
    kc, vc = (torch.randn(3 * M, Hkv, BS, D, dtype=dtype) for _ in range(2))
    bias = torch.randn(n, dtype=dtype) if M % 2 else None
    xss = (torch.rand(M, 12) * k / 6, k, 1e-5) if M != 8 else None
    to = lambda t: None if t is None else t.to(dev)      # noqa: E731
    return (n, fmt, blob, to(x), to(tab), to(pos), to(lens), to(bt), to(kc), to(vc), to(bias),
            None if xss is None else (to(xss[0]), *xss[1:]))


def _check(q, Hq, Hkv, D, k, M, dtype, dev):
    n, fmt, blob, x, tab, pos, lens, bt, kc, vc, bias, xss = _case(q, Hq, Hkv, D, k, M, dtype, dev)
    out = ops.gemv_rope(x, blob, fmt, n, k, bias, torch.empty(M, n, device=dev), (tab, pos, (Hq + Hkv) * D, D), xss=xss)
    wq, wk, wv = out.to(dtype).view(M, -1, D).split([Hq, Hkv, Hkv], 1)
    k1, v1 = kc.clone(), vc.clone()
    for m in range(M):
        at = int(lens[m]) - 1
        blk = int(bt[m, at // BS]) if 0 <= at < 3 * BS else -1
        if 0 <= blk < kc.shape[0]:
            k1[blk, :, at % BS], v1[blk, :, at % BS] = wk[m], wv[m]
    got = ops.gemv_rope_kv(x, blob, fmt, n, k, bias, tab, pos, kc, vc, bt, lens, Hq, xss=xss)
    assert got.shape == (M, Hq, D) and torch.equal(got, wq) and torch.equal(kc, k1) and torch.equal(vc, v1)


def test_on_the_host():
    _check("sym_int4", 4, 2, 64, 128, 9, torch.bfloat16, torch.device("cpu"))


@pytest.mark.gpu
@pytest.mark.parametrize("Hq,Hkv,D,k", [(4, 1, 128, 128), (7, 1, 64, 2048), (4, 2, 128, 4160), (2, 2, 64, 8320)])
@pytest.mark.parametrize("q", ["sym_int4", "asym_int4", "nf4", "sym_int8", "fp8_e5m2"])
def test_rows(cuda, q, Hq, Hkv, D, k):
    for M, dtype in ((1, torch.bfloat16), (3, torch.float16), (8, torch.bfloat16), (9, torch.bfloat16), (16, torch.float16)):
        _check(q, Hq, Hkv, D, k, M, dtype, cuda)


@pytest.mark.gpu
def test_refused(cuda):
    n, fmt, blob, x, tab, pos, lens, bt, kc, vc, bias, xss = _case("sym_int4", 4, 1, 128, 256, 3, torch.bfloat16, cuda)
    for bad in (dict(kc=kc.half()), dict(kc=kc[:, :, ::2]), dict(vc=vc[:-1]), dict(lens=lens[:2]), dict(lens=lens.long()), dict(bt=bt[:2]),
                dict(Hq=5), dict(bt=bt.t())):
        a = dict(kc=kc, vc=vc, bt=bt, lens=lens, Hq=4)
        a.update(bad)
        with pytest.raises(RuntimeError):
            ops.gemv_rope_kv(x, blob, fmt, n, 256, bias, tab, pos, a["kc"], a["vc"], a["bt"], a["lens"], a["Hq"], xss=xss)
