"""The product that finishes its rows (residual add, deferred-norm input, sums of squares by 16 columns) and the launches
that take its parts, against f64 over the dequantized weights.

Bounds: rounding to 16 bits moves a value by half a step at most, 2^-8 (bf16) or 2^-11 (f16) of itself, and the residual
add rounds the product first, hence two roundings; beside them the error of the 32-bit sums, 2^-18 of the sum of
magnitudes for the up to 2^11 additions of one of them, and of the f16 table of the table formats, whose entries are
2^-11 of themselves off at most."""
import pytest
import torch

import ipex_llm_amd.ops as ops
from ipex_llm_amd.quantize import qtypes as Q

pytestmark = pytest.mark.gpu

HALF = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}
# edges: one chunk, fewer chunks than waves, K inside a chunk, ends of a piece of 4 (2) chunks and of two pieces ahead (K of
# 4096, 4224, 8192, 8320, 12416 over 8 waves), a last tile of 4 columns, the widest K
SHAPES = [(64, 128), (64, 192), (132, 640), (64, 1088), (320, 2048), (64, 2176), (192, 4096), (64, 4224), (128, 8192),
          (64, 8320), (64, 12416), (64, 28672)]


def fmt_of(q):
    return Q.get_format(Q.resolve_qtype(q)).fmt


def make(q, n, k, M, dtype, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    fmt = fmt_of(q)
    blob = ops.quantize(torch.randn(n, k, device="cuda", generator=g) * 0.05, fmt)
    w = ops.dequantize(blob, fmt, n, k, torch.float32).double()
    r = lambda *s: torch.randn(*s, device="cuda", generator=g).to(dtype)        # noqa: E731
    return fmt, blob, w, r(M, k), r(M, n), r(n)


def check(q, n, k, M, dtype, unit=False, alone=True):
    fmt, blob, w, x, res, nw = make(q, n, k, M, dtype)
    NT = (n + 15) // 16
    full = torch.full((M + 2, n), 7.0, device="cuda", dtype=dtype)              # a row before and behind each output
    full2, ss = full.clone(), torch.full((M + 2, NT), 7.0, device="cuda")
    clear = torch.ones(M + 2, n, device="cuda")
    ops.gemv_row_norm(x, blob, fmt, n, k, res, full[1:-1], nw, unit, full2[1:-1], ss[1:-1], zero=clear[1:-1])
    for t in (full, full2, ss):
        assert (t[0] == 7).all() and (t[-1] == 7).all()
    assert (clear[1:-1] == 0).all() and (clear[0] == 1).all() and (clear[-1] == 1).all()
    h, xo, ss = full[1:-1], full2[1:-1], ss[1:-1]
    y = x.double() @ w.t()
    scale = (x.double().abs() @ w.abs().t())
    e = HALF[dtype]
    bound = (y.abs() + (y + res.double()).abs()) * e * 1.01 + scale * (2.0 ** -11 if q in ("nf4", "nf3") else 2.0 ** -18)
    assert ((h.double() - (y + res.double())).abs() <= bound).all()
    wv = (nw.double() + 1).to(dtype).double() if unit else nw.double()
    want = wv * h.double()
    assert ((xo.double() - want).abs() <= want.abs() * e * 1.001 + 1e-7).all()
    sq = torch.nn.functional.pad(h.double().pow(2), (0, -n % 16)).view(M, NT, 16).sum(-1)
    assert torch.allclose(ss.double(), sq, rtol=2e-6, atol=1e-12)
    # the same bits again, and with other rows beside a row
    h2, xo2, ss2 = torch.empty_like(h), torch.empty_like(h), torch.empty_like(ss)
    ops.gemv_row_norm(x, blob, fmt, n, k, res, h2, nw, unit, xo2, ss2)
    assert torch.equal(h, h2) and torch.equal(xo, xo2) and torch.equal(ss, ss2)
    if not alone:
        return
    h1, xo1, ss1 = h[-1:].clone(), xo[-1:].clone(), ss[-1:].clone()
    ops.gemv_row_norm(x[-1:], blob, fmt, n, k, res[-1:].clone(), h1, nw, unit, xo1, ss1)
    assert torch.equal(h1, h[-1:]) and torch.equal(xo1, xo[-1:]) and torch.equal(ss1, ss[-1:])


@pytest.mark.parametrize("n,k", SHAPES)
@pytest.mark.parametrize("q", ["sym_int4", "asym_int4", "fp8_e5m2"])
def test_shapes(n, k, q):
    for M in (1, 8, 9):
        check(q, n, k, M, torch.bfloat16, alone=not 8192 < k <= 16384)


# 16 waves: from a K of 8 chunks a wave on, two pieces each at most
@pytest.mark.parametrize("k", [8192, 8256, 14336, 16384, 16448])
@pytest.mark.parametrize("q", ["sym_int4", "asym_int4", "nf4", "fp4", "sym_int8", "asym_int5", "fp8_e5m2"])
def test_sixteen_waves(q, k):
    for M, dtype in ((1, torch.bfloat16), (2, torch.float16), (3, torch.bfloat16), (4, torch.bfloat16)):
        check(q, 48, k, M, dtype, alone=False)      # (a row's waves, so its sums, go by the number of rows here)


@pytest.mark.parametrize("q", ["sym_int4", "asym_int4", "nf4", "nf3", "fp4", "sym_int8", "sym_int5", "asym_int5",
                               "fp8_e4m3", "fp8_e5m2", "fp6"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_formats_and_rows(q, dtype):
    for M in (1, 2, 3, 4, 5, 8, 9, 16):
        check(q, 80, 4480, M, dtype, unit=M == 3)


def test_refused():
    fmt, blob, _, x, res, nw = make("sym_int4", 64, 256, 4, torch.bfloat16)
    ro, xo, ss = torch.empty_like(res), torch.empty_like(res), torch.empty(4, 4, device="cuda")
    ok = lambda **k: dict(dict(x=x, residual=res, res_out=ro, norm_w=nw, xo=xo, ss=ss), **k)   # noqa: E731

    def call(x, residual, res_out, norm_w, xo, ss):
        ops.gemv_row_norm(x, blob, fmt, 64, 256, residual, res_out, norm_w, False, xo, ss)
    call(**ok())
    for bad in (dict(res_out=res), dict(ss=ss[:, :3].contiguous()), dict(ss=ss.half()), dict(norm_w=nw.float()),
                dict(residual=res[:3]), dict(xo=xo.t()), dict(x=torch.cat([x] * 5))):
        with pytest.raises(RuntimeError):
            call(**ok(**bad))


@pytest.mark.parametrize("q,n,k", [("sym_int4", 1024, 512), ("fp8_e5m2", 512, 1024), ("nf4", 256, 512),
                                   ("sym_int4", 28672, 4096), ("asym_int4", 256, 1088)])
@pytest.mark.parametrize("M", [1, 3, 8, 16])
def test_consumers_add_the_parts(q, n, k, M):
    """gate/up (decode and skinny kernels) and the rotated qkv sums: the launch on parts against the one on whole sums"""
    fmt, blob, w, x, _, _ = make(q, n, k, M, torch.bfloat16, 1)
    parts = torch.rand(M, k // 16, device="cuda") * 16
    whole = parts.double().sum(-1)
    a = ops.gemv_glu_ss(x, blob, fmt, n, k, 0, parts, k, 1e-5, parts=True)
    b = ops.gemv_glu_ss(x, blob, fmt, n, k, 0, whole.float(), k, 1e-5)
    # both rounded to 16 bits, by half a step at most, from 32-bit sums in another order
    assert ((a.double() - b.double()).norm() / b.double().norm()).item() <= 2 * 2.0 ** -8 * 1.01
    if n > 4096:
        return
    D, cols = 128, n // 256 * 128
    tab = torch.randn(64, D // 2, 2, device="cuda")
    pos = torch.randint(0, 64, (M,), device="cuda")
    acc = torch.zeros(M, n, device="cuda")
    ops.gemv_accum(x, blob, fmt, n, k, acc, rope=(tab, pos, cols, D), xss=(parts, k, 1e-5))
    y = (x.double() @ w.t()) * torch.rsqrt(whole / k + 1e-5)[:, None]
    cs = tab[pos].to(torch.bfloat16).double()
    c, s = (torch.cat([cs[..., i]] * 2, -1)[:, None] for i in (0, 1))
    r = y[:, :cols].reshape(M, -1, D)
    y[:, :cols] = (r * c + torch.cat([-r[..., D // 2:], r[..., :D // 2]], -1) * s).reshape(M, cols)
    assert ((acc.double() - y).norm() / y.norm()).item() < (2e-3 if q == "nf4" else 1e-5)   # (an f16 table)


@pytest.mark.parametrize("M", [1, 4, 9])
def test_whole_sums_in_any_shape(M):
    """sums of squares that are not called parts are one a row, whatever the shape that holds them"""
    fmt, blob, _, x, _, _ = make("sym_int4", 256, 512, M, torch.bfloat16, 5)
    whole = torch.rand(M, device="cuda") * 512
    want = ops.gemv_glu_ss(x, blob, fmt, 256, 512, 0, whole, 512, 1e-5)
    more = torch.cat([whole, torch.rand(3 * M, device="cuda")])
    for ss in (whole[:, None], whole[None], more.view(M, 4), more.view(4, M)):
        assert torch.equal(ops.gemv_glu_ss(x, blob, fmt, 256, 512, 0, ss, 512, 1e-5), want)


def test_rule():
    """a down projection finishes its rows: 8 bits, integers in well-filled rounds; 4 bits of at most one workgroup per CU
    but for what row_norm_takes names; an o projection but for wide tables"""
    ops.require()
    f = lambda M, n, k, q: torch.ops.ipex_llm_amd.row_norm_takes(M, n, k, fmt_of(q))      # noqa: E731
    assert [f(M, 4096, 14336, "sym_int4") for M in (1, 2, 3, 8, 9, 16, 17)] == [True, True, False, False, True, True, False]
    assert [f(M, 4096, 14336, "nf4") for M in (1, 2, 3, 12, 13)] == [True, True, False, False, True]
    assert f(8, 3584, 18944, "sym_int4") and f(8, 8192, 28672, "fp8_e5m2") and f(4, 4096, 14336, "asym_int4")
    assert not f(1, 5120, 13824, "sym_int4")
    for q in ("sym_int8", "sym_int5", "asym_int5"):          # rounds of one workgroup per CU: the last at least half full
        assert [f(5, 16 * t, 13824, q) for t in (256, 257, 320, 383, 384, 512, 513)] == [True, False, False, False, True, True,
                                                                                          False]
    assert all(f(5, 5120, 13824, q) for q in ("fp8_e4m3", "fp8_e5m2", "fp6"))
    o = lambda M, n, q: torch.ops.ipex_llm_amd.row_norm_o_takes(M, n, fmt_of(q))          # noqa: E731
    for q in ("nf4", "nf3"):
        assert [o(M, 5120, q) for M in (1, 4, 5, 8)] == [True, True, False, False] and o(16, 4096, q) and not o(17, 4096, q)
    assert o(8, 5120, "sym_int4") and o(8, 8192, "fp4") and o(8, 8192, "sym_int8") and not o(17, 4096, "sym_int4")
    g = lambda M, n, k, q: torch.ops.ipex_llm_amd.row_norm_takes(M, n, k, fmt_of(q), True)      # noqa: E731
    assert g(8, 4096, 14336, "sym_int4") and g(8, 4096, 14336, "nf4") and not g(8, 5120, 13824, "sym_int4")
    r = lambda M, n, k, q: torch.ops.ipex_llm_amd.row_rope_takes(M, n, k, fmt_of(q))            # noqa: E731
    assert r(1, 6144, 4096, "sym_int4") and r(1, 10240, 8192, "fp8_e5m2") and r(16, 10240, 8192, "sym_int4")
    assert not r(8, 10240, 8192, "sym_int4") and not r(17, 6144, 4096, "sym_int4")


# heads of both sizes, a K of one chunk, of one and two pieces a wave and past them, tables' f16 entries (2^-11) beside 32-bit
# sums
@pytest.mark.parametrize("n,k,D,cols", [(384, 128, 128, 256), (192, 64, 64, 128), (768, 2048, 128, 640), (384, 4160, 128, 256),
                                        (512, 8320, 128, 384), (128, 4096, 64, 0)])
@pytest.mark.parametrize("q", ["sym_int4", "asym_int4", "nf4", "fp4", "sym_int8", "asym_int5", "fp8_e4m3", "fp8_e5m2"])
def test_rotated_rows(q, n, k, D, cols):
    for M, dtype in ((1, torch.bfloat16), (3, torch.float16), (8, torch.bfloat16), (9, torch.bfloat16), (16, torch.float16)):
        fmt, blob, w, x, _, _ = make(q, n, k, M, dtype, 2)
        tab = torch.randn(64, D // 2, 2, device="cuda")
        pos = torch.randint(0, 64, (M,), device="cuda")
        bias = torch.randn(n, device="cuda").to(dtype) if M != 3 else None
        parts = torch.rand(M, 12, device="cuda") * 16 if M != 8 else None
        out = torch.full((M + 2, n), 7.0, device="cuda")
        xss = None if parts is None else (parts, k, 1e-5)
        ops.gemv_rope(x, blob, fmt, n, k, bias, out[1:-1], (tab, pos, cols, D), xss=xss)
        assert (out[0] == 7).all() and (out[-1] == 7).all()
        y, mag = x.double() @ w.t(), x.double().abs() @ w.abs().t()
        if parts is not None:
            rs = torch.rsqrt(parts.double().sum(-1) / k + 1e-5)[:, None]
            y, mag = y * rs, mag * rs
        if bias is not None:
            y, mag = y + bias.double(), mag + bias.double().abs()
        cs = tab[pos].to(dtype).double()
        c, s = (torch.cat([cs[..., i]] * 2, -1)[:, None] for i in (0, 1))
        r, m = (t[:, :cols].reshape(M, -1, D) for t in (y.clone(), mag.clone()))
        half = lambda t: torch.cat([t[..., D // 2:], t[..., :D // 2]], -1)      # noqa: E731
        y[:, :cols] = (r * c + torch.cat([-r[..., D // 2:], r[..., :D // 2]], -1) * s).reshape(M, cols)
        mag[:, :cols] = (m * c.abs() + half(m) * s.abs()).reshape(M, cols)
        # codes of 4-bit integers carry an offset (f16 1032, bf16 136 beside values of up to 8: 140 and 18 times the largest
        # weight, for every x) until the block's sum is done: eight of its steps at most
        off = (140 if dtype == torch.float16 else 18) if q in ("sym_int4", "asym_int4") else 2
        big = x.double().abs().sum(-1, keepdim=True) * w.abs().amax(-1)[None] * off
        if parts is not None:
            big = big * rs
        if cols:
            b = big[:, :cols].reshape(M, -1, D)
            big[:, :cols] = (b * c.abs() + half(b) * s.abs()).reshape(M, cols)
        bound = mag * (2.0 ** -11 if q == "nf4" else 2.0 ** -18) + big * 2.0 ** -21
        assert ((out[1:-1].double() - y).abs() <= bound + 1e-7).all()
        a = torch.empty(1, n, device="cuda")                                    # the same bits without its neighbours
        ops.gemv_rope(x[-1:], blob, fmt, n, k, bias, a, (tab, pos[-1:].clone(), cols, D),
                      xss=None if xss is None else (parts[-1:].clone(), k, 1e-5))
        assert torch.equal(a, out[-2:-1])


@pytest.mark.parametrize("q", ["sym_int4", "fp8_e5m2"])
def test_columns_that_are_not_rotated_stand_alone(q):
    """an infinite value column says nothing of the column half a head away"""
    n, k, D, cols, M = 384, 256, 128, 256, 3
    fmt, blob, _, x, _, _ = make(q, n, k, M, torch.bfloat16, 6)
    tab, pos = torch.randn(64, D // 2, 2, device="cuda"), torch.randint(0, 64, (M,), device="cuda")
    bias = torch.zeros(n, device="cuda", dtype=torch.bfloat16)
    want, got = torch.empty(M, n, device="cuda"), torch.empty(M, n, device="cuda")
    ops.gemv_rope(x, blob, fmt, n, k, bias, want, (tab, pos, cols, D))
    at = [cols + 5, cols + 70, cols + 127]
    bias[at] = torch.tensor([float("inf"), -float("inf"), float("nan")], device="cuda").to(torch.bfloat16)
    ops.gemv_rope(x, blob, fmt, n, k, bias, got, (tab, pos, cols, D))
    assert (got[:, at[0]] == float("inf")).all() and (got[:, at[1]] == -float("inf")).all() and got[:, at[2]].isnan().all()
    rest = [c for c in range(n) if c not in at]
    assert torch.equal(got[:, rest], want[:, rest])


# one chunk, chunks for some waves only, one piece a wave; M <= 8 on the product that finishes its rows, then the others
@pytest.mark.parametrize("n,k", [(64, 128), (96, 576), (1024, 2048), (160, 4096), (64, 4160), (28672, 512)])
@pytest.mark.parametrize("q", ["sym_int4", "asym_int4", "nf4", "fp4", "sym_int8", "asym_int5", "fp8_e4m3", "fp8_e5m2"])
def test_gate_up_rows(q, n, k):
    for M, dtype, act in ((1, torch.bfloat16, 0), (2, torch.float16, 1), (5, torch.bfloat16, 1), (8, torch.bfloat16, 0),
                          (9, torch.bfloat16, 0)):
        fmt, blob, w, x, _, _ = make(q, n, k, M, dtype, 3)
        parts = torch.rand(M, 8, device="cuda") * k / 4
        got = ops.gemv_glu_ss(x, blob, fmt, n, k, act, parts, k, 1e-5, parts=True)
        y = (x.double() @ w.t()) * torch.rsqrt(parts.double().sum(-1) / k + 1e-5)[:, None]
        g, u = y.view(M, n // 32, 2, 16).unbind(2)
        f = torch.nn.functional.silu(g) if act == 0 else torch.nn.functional.gelu(g, approximate="tanh")
        want = (f * u).reshape(M, n // 2)
        assert got.shape == want.shape
        # every value rounded, by half a step of itself at most, from 32-bit sums, and the tables' entries
        rel = ((got.double() - want).norm() / want.norm()).item()
        assert rel <= HALF[dtype] + (2.0 ** -10 if q == "nf4" else 2.0 ** -16), (M, rel)


@pytest.mark.parametrize("B", [1, 5, 8, 9, 16, 17])
@pytest.mark.parametrize("q,bias", [("sym_int4", True), ("fp8_e5m2", False)])
def test_step_of_many_sequences(B, q, bias):
    """a decode step on either side of every rule by rows, captured and replayed, against the same step in f32"""
    from transformers import LlamaConfig, Qwen2Config
    from ipex_llm_amd.engine.runner import Engine
    from ipex_llm_amd.models.builder import random_native_model
    import __graft_entry__ as G
    dev = torch.device("cuda")
    cfg = (Qwen2Config if bias else LlamaConfig)(vocab_size=512, hidden_size=1024, intermediate_size=2560,
                                                 num_hidden_layers=3, num_attention_heads=8, num_key_value_heads=2,
                                                 max_position_embeddings=512)
    torch.manual_seed(1)
    m = random_native_model(cfg, q, dev, torch.bfloat16, seed=0)
    if bias:
        for L in m.layers:
            qkv = L.self_attn.qkv_proj
            qkv.bias = torch.nn.Parameter(torch.randn(qkv.out_features, device=dev, dtype=torch.bfloat16) * 0.2, False)
    eng = Engine(m)
    n, steps = 40, 3
    eng._ensure_cache(B, 64)
    seqs = [eng.new_sequence(64) for _ in range(B)]
    prompts = torch.randint(0, 512, (B, n), generator=torch.Generator().manual_seed(7))
    eng.prefill_batch(seqs, prompts)
    st = eng.decode_step_obj(seqs, 64, False, True)
    toks = torch.randint(0, 512, (B, steps), generator=torch.Generator().manual_seed(8))
    got = []
    st.set_state(toks[:, 0].to(dev), torch.full((B,), n, device=dev))
    for i in range(steps):
        st.ids.copy_(toks[:, i])
        st.step()
        got.append(st.logits.float().cpu().clone())
    W = [L.self_attn.qkv_proj.bias for L in m.layers]
    for b in {0, B - 1}:
        ref = _reference(m, torch.cat([prompts[b], toks[b]]), W, G)[n:n + steps]
        out = torch.stack([g[b] for g in got])
        assert ((out - ref).norm() / ref.norm()).item() < 3e-2      # 16-bit activations through three layers, as smoke()


@pytest.mark.parametrize("B", [9, 16])
@pytest.mark.parametrize("q,dtype", [("sym_int4", torch.float16), ("nf4", torch.bfloat16), ("sym_int4", torch.bfloat16)])
def test_large_residual_channel(B, q, dtype):
    """a channel of the residual stream of 3e4 under a norm weight of 4: past what f16 holds before the norm's scale,
    ordinary behind it.  The final norm leaves that channel out, so the logits are the layers' work"""
    from transformers import LlamaConfig
    from ipex_llm_amd.engine.runner import Engine
    from ipex_llm_amd.models.builder import random_native_model
    import __graft_entry__ as G
    dev = torch.device("cuda")
    cfg = LlamaConfig(vocab_size=512, hidden_size=1024, intermediate_size=2560, num_hidden_layers=3, num_attention_heads=8,
                      num_key_value_heads=2, max_position_embeddings=512)
    m = random_native_model(cfg, q, dev, dtype, seed=3)
    m.embed_tokens.data[:, 77] = 3e4
    for L in m.layers:
        L.input_layernorm.data[77] = L.post_attention_layernorm.data[77] = 4.0
    m.norm.data[77] = 0.0
    eng, n, steps = Engine(m), 20, 2
    eng._ensure_cache(B, 64)
    seqs = [eng.new_sequence(64) for _ in range(B)]
    ids = torch.randint(0, 512, (B, n + steps), generator=torch.Generator().manual_seed(9))
    eng.prefill_batch(seqs, ids[:, :n])
    st = eng.decode_step_obj(seqs, 64, False, True)
    st.set_state(ids[:, n].to(dev), torch.full((B,), n, device=dev))
    for i in range(steps):
        st.ids.copy_(ids[:, n + i])
        st.step()
        got = st.logits.float().cpu()
        for b in {0, B - 1}:
            ref = G._fp32_reference(m, ids[b, :n + i + 1])[-1]
            assert ((got[b] - ref).norm() / ref.norm()).item() < 3e-2       # 16-bit activations, as above


def _steps(m, B, first):
    """logits of two eager steps behind the same prompts"""
    from ipex_llm_amd.engine.runner import Engine
    eng = Engine(m)
    eng._ensure_cache(B, 64)
    seqs = [eng.new_sequence(64) for _ in range(B)]
    ids = torch.randint(0, 512, (B, 22), generator=torch.Generator().manual_seed(4))
    eng.prefill_batch(seqs, ids[:, :20])
    st = eng.decode_step_obj(seqs, 64, False, False)
    st.set_state(ids[:, 20].cuda(), torch.full((B,), 20, device="cuda"))
    out = []
    for i in range(2):
        st.ids.copy_(ids[:, 20 + i])
        st.step()
        out.append(st.logits.float().clone())
        if i == 0:
            first()
    return torch.stack(out)


@pytest.mark.parametrize("what", ["dense_o", "dense_qkv", "oproj_combine", "row_norm_off"])
@pytest.mark.parametrize("B", [2, 9])
def test_model_that_changes_between_steps(B, what, monkeypatch):
    """a projection replaced or a launch switched after a step: the next step goes by what is there"""
    import ipex_llm_amd.models.decoder as D
    from transformers import LlamaConfig
    from ipex_llm_amd.models.builder import random_native_model
    cfg = LlamaConfig(vocab_size=512, hidden_size=1024, intermediate_size=2560, num_hidden_layers=3, num_attention_heads=8,
                      num_key_value_heads=2, max_position_embeddings=512)
    m = random_native_model(cfg, "sym_int4", torch.device("cuda"), torch.bfloat16, seed=0)
    want = _steps(m, B, lambda: None)

    def dense(mod):
        lin = torch.nn.Linear(mod.in_features, mod.out_features, bias=False, device="meta")
        lin.weight = torch.nn.Parameter(mod.dequantize(torch.float32).to("cuda", torch.bfloat16), False)
        return lin

    def change():
        L = m.layers[1]
        if what == "dense_o":
            L.self_attn.o_proj = dense(L.self_attn.o_proj)
        elif what == "dense_qkv":
            L.self_attn.qkv_proj = dense(L.self_attn.qkv_proj)
        elif what == "oproj_combine":
            monkeypatch.setattr(D.NativeCausalLM, "_oproj_combine", True)
        else:
            monkeypatch.setattr(D, "ROW_NORM", False)
    got = _steps(m, B, change)
    for g, w in zip(got, want):
        assert ((g - w).norm() / w.norm()).item() < 2e-2        # 16-bit activations, rounded at other places


def _reference(m, ids, biases, G):
    """``__graft_entry__``'s f32 forward with the qkv bias"""
    if biases[0] is None:
        return G._fp32_reference(m, ids)
    import torch.nn.functional as F
    from ipex_llm_amd.models.decoder import deinterleave_glu
    s = m.spec

    def rms(x, w):
        return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + s.rms_eps) * w.float().cpu()
    T = ids.shape[0]
    x = m.embed_tokens.float().cpu()[ids]
    fr = torch.arange(T, dtype=torch.float32)[:, None] * m.inv_freq.float().cpu()[None]
    cos, sin = torch.cat([fr.cos()] * 2, -1), torch.cat([fr.sin()] * 2, -1)

    def rope(t):
        a, b = t.chunk(2, -1)
        return t * cos[:, None] + torch.cat([-b, a], -1) * sin[:, None]
    nh, nkv, hd = s.num_heads, s.num_kv_heads, s.head_dim
    W = lambda mod: mod.dequantize(torch.float32).cpu()              # noqa: E731
    for L in m.layers:
        qkv = rms(x, L.input_layernorm) @ W(L.self_attn.qkv_proj).t() + L.self_attn.qkv_proj.bias.float().cpu()
        q, k, v = qkv.split([nh * hd, nkv * hd, nkv * hd], -1)
        q, k, v = rope(q.view(T, nh, hd)), rope(k.view(T, nkv, hd)), v.view(T, nkv, hd)
        k, v = k.repeat_interleave(nh // nkv, 1), v.repeat_interleave(nh // nkv, 1)
        o = F.scaled_dot_product_attention(q.transpose(0, 1), k.transpose(0, 1), v.transpose(0, 1), is_causal=True,
                                           scale=s.scale)
        x = x + o.transpose(0, 1).reshape(T, -1) @ W(L.self_attn.o_proj).t()
        g, u = deinterleave_glu(rms(x, L.post_attention_layernorm) @ W(L.mlp.gate_up_proj).t())
        x = x + (F.silu(g) * u) @ W(L.mlp.down_proj).t()
    return rms(x, m.norm) @ W(m.lm_head).t()
