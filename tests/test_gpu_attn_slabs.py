"""Decode attention over the slabs of the qkv product (attn_decode_slabs): bit for bit rope_kv_fused and attn_decode, in the
output and in the caches -- one to six slabs, items of one pass over the workgroup and of several, the new key at the edges of
tiles and of a workgroup's, offsets of a compressed cache, padding rows, bad blocks -- and in a model's step, captured too."""
import pytest
import torch

import ipex_llm_amd.ops as ops

pytestmark = pytest.mark.gpu
T = torch.ops.ipex_llm_amd


def _both(dev, dtype, L, cap, Hkv, G, bs, ks, bias, window, offset, tables=None):
    torch.manual_seed(len(L) * cap + ks)
    B, Hq, D, nb = len(L), Hkv * G, 128, -(-cap // bs)
    kc, vc = (torch.randn(nb * B, Hkv, bs, D, device=dev).to(dtype) for _ in range(2))
    bt = torch.randperm(nb * B, device=dev).int().view(B, nb).contiguous()
    if tables is not None:
        tables(bt)
    sl, ns = torch.tensor(L, dtype=torch.int32, device=dev), -(-cap // 64)
    off = torch.arange(B, device=dev) * 3 if offset else None
    pos = (sl.long() - 1).clamp(min=0) + (off if offset else 0)
    cs = torch.randn(cap + 3 * B, D // 2, 2, device=dev)
    part = torch.randn(ks, B, (Hq + 2 * Hkv) * D, device=dev)
    b = torch.randn((Hq + 2 * Hkv) * D, device=dev).to(dtype) if bias else None
    k1, v1, q = kc.clone(), vc.clone(), torch.empty(B, Hq, D, dtype=dtype, device=dev)
    ops.rope_kv_fused(part, b, q, k1, v1, pos, bt, 1, cs, Hq, Hkv, D, pos_offset=off)
    want = ops.attn_decode(q.view(B, 1, Hq, D), k1, v1, bt, sl, ns, D ** -0.5, 0.0, window)
    assert T.attn_slabs_takes(B, Hkv, ns)
    keep = part.clone()
    got = ops.attn_decode_slabs(part, b, cs, pos, off, kc, vc, bt, sl, ns, D ** -0.5, 0.0, window, Hq, dtype)
    assert torch.equal(part, keep)
    return want.view(B, -1), got.view(B, -1), (k1, v1), (kc, vc)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("L,cap,Hkv,G,bs", [
    ([1, 31, 32, 33, 127, 128, 129, 255, 256, 257, 511, 512, 513, 640, 639, 2, 64], 640, 8, 4, 64),
    ([1, 128, 129, 256, 257, 513, 640, 31, 32, 33] * 4, 640, 8, 7, 128),
    ([1, 32, 129, 191, 192] * 2, 192, 8, 16, 192),
    ([511, 33, 1] * 3, 512, 2, 1, 64),
    ([3072, 1, 1024, 1025, 2048, 2049, 33, 3000, 1023] * 2, 3072, 8, 4, 64),   # several workgroups a pair
    ([1345, 1, 1024, 1025] * 10, 1408, 8, 7, 128),
])
@pytest.mark.parametrize("ks,bias,window,offset", [(1, True, 0, False), (2, False, 0, False), (4, True, 100, True), (6, False, 0, True)])
def test_same_bits(cuda, dtype, L, cap, Hkv, G, bs, ks, bias, window, offset):
    want, got, old, new = _both(cuda, dtype, L, cap, Hkv, G, bs, ks, bias, window, offset)
    ops.check_kernel_errors(cuda)
    assert torch.equal(got, want) and all(torch.equal(a, b) for a, b in zip(old, new))


@pytest.mark.parametrize("cap", [128, 3072])                       # one workgroup a pair, three
def test_padding_rows_and_bad_blocks(cuda, cap):
    L = [0, 100, 64, 65, 7, cap] * 3

    def padded(bt):
        bt[0] = -1
    want, got, old, new = _both(cuda, torch.bfloat16, L, cap, 8, 4, 64, 2, False, 0, False, padded)
    ops.check_kernel_errors(cuda)
    assert torch.equal(got, want) and all(torch.equal(a, b) for a, b in zip(old, new))

    def bad(bt):
        bt[1, 1] = bt[5, -1] = bt.numel() + 5
    want, got, old, new = _both(cuda, torch.bfloat16, L, cap, 8, 4, 64, 2, False, 0, False, bad)
    with pytest.raises(RuntimeError):
        ops.check_kernel_errors(cuda)
    assert torch.equal(got, want) and all(torch.equal(a, b) for a, b in zip(old, new))


def test_not_taken(cuda):
    """several workgroups a pair in turn, and widths that are not the heads'"""
    assert not T.attn_slabs_takes(1, 8, 100)
    x = torch.zeros(2, 1, 6144, device=cuda)
    kc = torch.zeros(100, 8, 64, 128, dtype=torch.bfloat16, device=cuda)
    i = torch.zeros(1, 100, dtype=torch.int32, device=cuda)
    args = (None, torch.zeros(8, 64, 2, device=cuda), i[0, :1].long(), None, kc, kc.clone(), i, i[0, :1].contiguous())
    with pytest.raises(RuntimeError):
        ops.attn_decode_slabs(x, *args, 100, 0.1, 0.0, 0, 32, torch.bfloat16)
    with pytest.raises(RuntimeError):
        ops.attn_decode_slabs(x, *args, 1, 0.1, 0.0, 0, 16, torch.bfloat16)


def test_arguments_that_do_not_fit_are_refused(cuda):
    """what the launch would read as another type, past its end or on another device"""
    B, Hkv, Hq, bf = 17, 8, 32, torch.bfloat16
    part, cs = torch.zeros(2, B, 6144, device=cuda), torch.zeros(64, 64, 2, device=cuda)
    kc = torch.zeros(B, Hkv, 64, 128, dtype=bf, device=cuda)
    bt, sl = torch.arange(B, dtype=torch.int32, device=cuda).view(B, 1), torch.ones(B, dtype=torch.int32, device=cuda)
    good = dict(part=part, bias=torch.zeros(6144, dtype=bf, device=cuda), cos_sin=cs, pos=torch.zeros(B, dtype=torch.long, device=cuda),
                pos_offset=torch.zeros(B, dtype=torch.long, device=cuda), k_cache=kc, v_cache=kc.clone(), block_tables=bt, seq_lens=sl)
    rest = (1, 0.1, 0.0, 0, Hq, bf)
    ops.attn_decode_slabs(*good.values(), *rest)
    bad = [("bias", good["bias"].float()), ("bias", good["bias"].half()), ("bias", good["bias"][:6143].clone()), ("bias", good["bias"][:0]),
           ("bias", torch.zeros(12288, dtype=bf, device=cuda)[::2]), ("block_tables", bt[:, :0]), ("block_tables", bt[:16].contiguous()),
           ("block_tables", bt.flatten()), ("block_tables", bt.long()), ("seq_lens", sl[:16]), ("pos", good["pos"].int()),
           ("pos_offset", good["pos_offset"][:16])]
    bad += [(k, v.cpu()) for k, v in good.items() if k != "part"]
    for name, value in bad:
        with pytest.raises(RuntimeError):
            ops.attn_decode_slabs(*{**good, name: value}.values(), *rest)
    ops.check_kernel_errors(cuda)


def test_replays_of_a_long_grid(cuda):
    """several workgroups a pair, captured: the tickets are left as they were, whichever sequences are long in a replay"""
    torch.manual_seed(7)
    B, Hkv, Hq, D, cap, bf = 18, 8, 32, 128, 3072, torch.bfloat16
    kc, vc = (torch.randn(B * 48, Hkv, 64, D, device=cuda).to(bf) for _ in range(2))
    bt, cs = torch.arange(B * 48, dtype=torch.int32, device=cuda).view(B, 48), torch.randn(cap, D // 2, 2, device=cuda)
    part, sl, pos = torch.randn(2, B, 6144, device=cuda), torch.ones(B, dtype=torch.int32, device=cuda), torch.zeros(B, dtype=torch.long, device=cuda)
    k1, v1, q = kc.clone(), vc.clone(), torch.empty(B, Hq, D, dtype=bf, device=cuda)
    run = lambda: ops.attn_decode_slabs(part, None, cs, pos, None, kc, vc, bt, sl, 48, 0.1, 0.0, 0, Hq, bf)  # noqa: E731
    run()
    k1.copy_(kc), v1.copy_(vc)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = run()
    for step in range(6):
        L = torch.tensor([[1, 3072, 1024, 1025, 200, 2049][(b + step) % 6] for b in range(B)])
        sl.copy_(L), pos.copy_(L - 1), part.normal_()
        graph.replay()
        ops.rope_kv_fused(part, None, q, k1, v1, pos, bt, 1, cs, Hq, Hkv, D)
        want = ops.attn_decode(q.view(B, 1, Hq, D), k1, v1, bt, sl, 48, 0.1)
        assert torch.equal(out.view(B, -1), want.view(B, -1)) and torch.equal(k1, kc) and torch.equal(v1, vc)
    ops.check_kernel_errors(cuda)


@pytest.mark.parametrize("kind,qtype", [("llama", "sym_int4"), ("qwen2", "fp8_e5m2"), ("mistral", "nf4")])
@pytest.mark.parametrize("B", [11, 17, 64])
def test_model_step(cuda, kind, qtype, B, monkeypatch):
    from transformers import LlamaConfig, MistralConfig, Qwen2Config
    from ipex_llm_amd.engine.runner import nsplit_for
    from ipex_llm_amd.models.builder import random_native_model
    from ipex_llm_amd.models.decoder import AttnMeta
    kw = dict(vocab_size=512, hidden_size=1024, intermediate_size=768, num_hidden_layers=2, num_attention_heads=8,
              num_key_value_heads=2, max_position_embeddings=1024)
    cfg = {"llama": lambda: LlamaConfig(**kw), "qwen2": lambda: Qwen2Config(**kw),
           "mistral": lambda: MistralConfig(sliding_window=16, **kw)}[kind]()
    model = random_native_model(cfg, qtype, cuda, torch.bfloat16, seed=1)
    inner, calls = ops.attn_decode_slabs, []
    monkeypatch.setattr(ops, "attn_decode_slabs", lambda *a: (calls.append(1), inner(*a))[1])

    def step(on):
        cache = model.make_cache(128, batch=B)
        g = torch.Generator(device=cuda).manual_seed(B)
        for t in (*cache.k, *cache.v):
            t.normal_(generator=g)
        ids = torch.randint(0, 512, (B,), generator=g, device=cuda)
        pos = torch.arange(B, device=cuda) * 7 % 128
        bt = torch.arange(B * 2, device=cuda, dtype=torch.int32).view(B, 2)
        slots = bt.long()[torch.arange(B, device=cuda), pos // 64] * 64 + pos % 64
        meta = AttnMeta(B, 1, bt, (pos + 1).int(), nsplit_for(128))
        monkeypatch.setattr(type(model), "_rope_in_env", on)
        with torch.no_grad():
            out = model.forward_tokens(ids, pos, slots, meta, cache)
            if not on:
                return out, cache
            model.forward_tokens(ids, pos, slots, meta, cache)
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                cap = model.forward_tokens(ids, pos, slots, meta, cache)
            for _ in range(3):
                cap.zero_()
                graph.replay()
                assert torch.equal(cap, out)
                torch.cuda.synchronize()
        return out, cache
    want, c0 = step(False)
    assert not calls
    got, c1 = step(True)
    # (up to 16 sequences whose launches finish their rows have their own)
    rows = B <= 16 and qtype != "nf4"
    assert len(calls) == (0 if rows else 2 * 3)
    ops.check_kernel_errors(cuda)
    if not rows:
        assert torch.equal(got, want) and all(torch.equal(a, b) for a, b in zip((*c0.k, *c0.v), (*c1.k, *c1.v)))
