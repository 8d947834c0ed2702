"""The work that users of this library have it do, as measured cases.

Three kinds, each through the library's public entry points:

* ``decode``: one generated token for every running sequence -- ``Engine.decode_step_obj`` + ``DecodeStep.step``
  (the captured step that ``generate`` and ``bench.py`` replay), from a single chat to a serving batch, over
  contexts of every length;
* ``prefill``: the first token of new prompts -- ``Engine.prefill`` for one prompt (what ``generate`` calls),
  ``Engine.prefill_batch`` for several of one length;
* ``train``: one forward + backward of QLoRA fine-tuning -- ``optimize_model`` + ``get_peft_model`` over a decoder
  stack, the library's attention and its fused head + loss.

Models and sizes are those of ``bench.py`` and ``tools/bench_qlora.py``: Llama-3-8B, Qwen2.5-7B, random weights quantized
on the GPU.  The projections back into the residual stream are drawn smaller with the depth and the embedding at unit
spread, as models are initialised: a stack of equally large random layers amplifies the last bit of its 16-bit
activations into per cents.  Every weight lies on the grid of its format, so that what is stored is known here.
Weights, prompts and cached keys / values follow from the seed alone.
"""
from __future__ import annotations

import math
from types import SimpleNamespace

import torch
import torch.nn as nn
import torch.nn.functional as F
import torch.utils.checkpoint

DEV = "cuda"
BLOCK = 64                     # tokens per cache block
KV_STD = 1.28                  # spread of keys / values behind 0.02-spread weights of a 4096-wide model

MODELS = {
    "llama3-8b": dict(model_type="llama", vocab_size=128256, hidden_size=4096, intermediate_size=14336,
                      num_hidden_layers=32, num_attention_heads=32, num_key_value_heads=8,
                      max_position_embeddings=131072, rms_norm_eps=1e-5, rope_theta=500000.0),
    "qwen2.5-7b": dict(model_type="qwen2", vocab_size=152064, hidden_size=3584, intermediate_size=18944,
                       num_hidden_layers=28, num_attention_heads=28, num_key_value_heads=4,
                       max_position_embeddings=32768, rms_norm_eps=1e-6, rope_theta=1000000.0),
}
BITS = {"sym_int4": 4.25, "nf4": 4.25, "asym_int4": 4.5, "sym_int8": 8.25, "fp8_e5m2": 8.25}


def listed():
    d = dict(kind="decode", model="llama3-8b", qtype="sym_int4")
    p = dict(kind="prefill", model="llama3-8b", qtype="sym_int4")
    return [
        # a chat with one user: every token waits for one pass over the weights
        dict(d, name="decode_chat", batch=1, context=1024),
        # the default batch of bench.py
        dict(d, name="decode_batch8", batch=8, context=1024),
        # a serving engine under load: many sequences of different lengths
        dict(d, name="decode_serving", batch=48, context=700),
        # a long document: the cached keys weigh as much as the weights
        dict(d, name="decode_document", batch=3, context=20000),
        # the serving guide's model and 8-bit format (group of 7 query heads, qkv bias)
        dict(kind="decode", model="qwen2.5-7b", qtype="fp8_e5m2", name="decode_fp8", batch=5, context=777),
        # a chat turn: a short question, first token as soon as may be
        dict(p, name="prefill_short", batch=1, prompt=45),
        # a question with some context, the serving guide's model and format
        dict(kind="prefill", model="qwen2.5-7b", qtype="fp8_e5m2", name="prefill_fp8", batch=1, prompt=300),
        # the published 1024-token prompt
        dict(p, name="prefill_1k", batch=1, prompt=1024),
        # bench.py's batch of prompts
        dict(p, name="prefill_batch", batch=8, prompt=1024),
        # QLoRA fine-tuning at the recipe's batch (layers cut: every layer is alike)
        dict(kind="train", name="qlora_step", qtype="nf4", layers=4, batch=8, seq=512, rank=8),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["decode", "prefill", "train"], [0.5, 0.35, 0.15])[0]
    if kind == "train":
        batch = _log(rng, 1, 8)
        return dict(kind="train", qtype=rng.choice(["nf4", "sym_int4"]), layers=rng.randint(2, 4), batch=batch,
                    seq=64 * rng.randint(2, min(16, 64 // batch)), rank=rng.choice([8, 16]))
    c = dict(kind=kind, model=rng.choices(list(MODELS), [0.7, 0.3])[0],
             qtype=rng.choices(list(BITS), [0.5, 0.1, 0.1, 0.1, 0.2])[0])
    if kind == "decode":
        c["batch"] = _log(rng, 1, 64)
        c["context"] = _log(rng, 64, min(20000, 60000 // c["batch"]))
    else:
        c["batch"] = rng.choices([1, _log(rng, 2, 8)], [0.7, 0.3])[0]
        c["prompt"] = _log(rng, 17, min(2048, 6000 // c["batch"]))
    return c


# ------------------------------------------------------------ weights
class Weights:
    """the model's weights in the order of the layers: 16-bit vectors, matrices [n, k] on their format's grid"""

    def __init__(self, cfg, layers, qtype, seed):
        self.cfg, self.layers, self.qtype = cfg, layers, qtype
        self.dim = cfg.hidden_size // cfg.num_attention_heads
        self.g = torch.Generator(device=DEV).manual_seed(seed)

    def normal(self, *shape, std=0.02):
        return torch.empty(shape, dtype=torch.bfloat16, device=DEV).normal_(0, std, generator=self.g)

    def grid(self, n, k, std=0.02):
        w = torch.empty(n, k, dtype=torch.float32, device=DEV).normal_(0, std, generator=self.g)
        return _grid(w, self.qtype)

    def embed(self):
        return self.normal(self.cfg.vocab_size, self.cfg.hidden_size, std=1.0)

    def norm(self):
        return (1.0 + self.normal(self.cfg.hidden_size).float()).to(torch.bfloat16)

    def layer(self):
        c, H, D = self.cfg, self.cfg.hidden_size, self.dim
        back = 0.02 / math.sqrt(2 * self.layers)
        w = {n: self.grid(h * D, H) for n, h in (("q", c.num_attention_heads), ("k", c.num_key_value_heads),
                                                 ("v", c.num_key_value_heads))}
        w["o"] = self.grid(H, c.num_attention_heads * D, back)
        w["gate"], w["up"] = self.grid(c.intermediate_size, H), self.grid(c.intermediate_size, H)
        w["down"] = self.grid(H, c.intermediate_size, back)
        if c.model_type == "qwen2":
            w["bias"] = self.normal((c.num_attention_heads + 2 * c.num_key_value_heads) * D, std=0.5)
        w["norm1"], w["norm2"] = self.norm(), self.norm()
        return w


_NF4 = [-1.0, -0.6961928009986877, -0.5250730514526367, -0.39491748809814453, -0.28444138169288635,
        -0.18477343022823334, -0.09105003625154495, 0.0, 0.07958029955625534, 0.16093020141124725,
        0.24611230194568634, 0.33791524171829224, 0.44070982933044434, 0.5626170039176941, 0.7229568362236023, 1.0]


def _grid(w, qtype):
    """``w`` [n, k] f32 moved to values that block quantization (64 values to a 16-bit scale) keeps as they are"""
    x = w.view(-1, 64)
    amax = x.abs().amax(-1, keepdim=True)
    if qtype == "sym_int4":                      # the value of the largest magnitude is code -8
        at = x.abs().argmax(-1, keepdim=True)
        d = (x.gather(-1, at) / -8).half().float()
        return (x.div_(d).round_().clamp_(-8, 7).scatter_(-1, at, -8.0) * d).view(w.shape)
    if qtype == "asym_int4":
        lo = x.amin(-1, keepdim=True)
        d = ((x.amax(-1, keepdim=True) - lo) / 15).half().float()
        return (x.sub_(lo).div_(d).round_().clamp_(0, 15) * d + lo.half().float()).view(w.shape)
    if qtype == "sym_int8":
        d = (amax / 127).half().float()
        return (x.div_(d).round_().clamp_(-127, 127) * d).view(w.shape)
    if qtype == "fp8_e5m2":
        at = x.abs().argmax(-1, keepdim=True)
        top = 57344 * x.gather(-1, at).sign()
        d = (amax / 57344).half().float()
        code = x.div_(d).clamp_(-57344, 57344).to(torch.float8_e5m2).float()
        return (code.scatter_(-1, at, top) * d).view(w.shape)
    d = amax.half().float()
    tab = torch.tensor(_NF4, device=x.device)
    return (tab[torch.bucketize(x.div_(d), (tab[1:] + tab[:-1]) / 2)] * d).view(w.shape)


# ------------------------------------------------------------ prepare
def _config(case):
    return SimpleNamespace(**MODELS[case.get("model", "llama3-8b")])


def _model(cfg, qtype, seed):
    from ipex_llm_amd.models.builder import lowbit_from_dense, spec_from_config
    from ipex_llm_amd.models.decoder import (NativeAttention, NativeCausalLM, NativeLayer, NativeMLP,
                                             compute_inv_freq, interleave_glu_rows)
    spec, W = spec_from_config(cfg), Weights(cfg, cfg.num_hidden_layers, qtype, seed)
    embed, layers = W.embed(), []
    for _ in range(cfg.num_hidden_layers):
        w = W.layer()
        attn = NativeAttention(spec, lowbit_from_dense(torch.cat([w["q"], w["k"], w["v"]]), qtype, DEV, w.get("bias")),
                               lowbit_from_dense(w["o"], qtype, DEV))
        mlp = NativeMLP(spec, lowbit_from_dense(interleave_glu_rows(w["gate"], w["up"]), qtype, DEV),
                        lowbit_from_dense(w["down"], qtype, DEV))
        layers.append(NativeLayer(spec, attn, mlp, w["norm1"], w["norm2"]))
    head, last = lowbit_from_dense(W.grid(cfg.vocab_size, cfg.hidden_size), qtype, DEV), W.norm()
    inv, spec.rope_attention_scaling = compute_inv_freq(cfg, spec.head_dim, spec.rot_dim)
    return NativeCausalLM(spec, embed, layers, last, head, inv.to(DEV), torch.bfloat16).eval()


@torch.no_grad()
def prepare(case, seed):
    if case["kind"] == "train":
        return _prepare_train(case, seed)
    from ipex_llm_amd.engine.runner import Engine
    from ipex_llm_amd.models.cache import SequenceState
    cfg, B = _config(case), case["batch"]
    eng = Engine(_model(cfg, case["qtype"], seed))
    most = case["context"] + BLOCK if case["kind"] == "decode" else case["prompt"] + BLOCK
    nblk = -(-most // BLOCK)
    eng._ensure_cache(B, nblk * BLOCK)
    seqs = [SequenceState(eng.cache.allocator.alloc(nblk)) for _ in range(B)]
    if case["kind"] == "prefill":
        ids = _tokens(case, seed, cfg.vocab_size)
        return dict(kind="prefill", eng=eng, seqs=seqs, ids=ids if B > 1 else ids[0])
    ids, lens = _next_tokens(case, seed, cfg.vocab_size)
    step = eng.decode_step_obj(seqs, nblk * BLOCK, greedy=True, use_graph=True)
    rows = torch.tensor([b for s in seqs for b in s.blocks], device=DEV)
    for li, (k, v) in enumerate(_cached(case, seed, cfg)):
        eng.cache.k[li][rows] = k
        eng.cache.v[li][rows] = v
    return dict(kind="decode", eng=eng, step=step, ids=ids.to(DEV), pos=lens.to(DEV))


def _tokens(case, seed, vocab):
    g = torch.Generator().manual_seed(seed + 1)
    return torch.randint(0, vocab, (case["batch"], case["prompt"]), generator=g)


def _next_tokens(case, seed, vocab):
    """a token and a number of cached tokens (half the context to all of it) for every sequence"""
    g = torch.Generator().manual_seed(seed + 1)
    ids = torch.randint(0, vocab, (case["batch"],), generator=g)
    n = case["context"]
    return ids, torch.randint(n // 2, n + 1, (case["batch"],), generator=g)


def _cached(case, seed, cfg):
    """(keys, values) of every layer, block by block and sequence after sequence: [blocks, kv heads, 64, head dim]"""
    g = torch.Generator(device=DEV).manual_seed(seed + 2)
    n = case["batch"] * -(-(case["context"] + BLOCK) // BLOCK)
    shape = (n, cfg.num_key_value_heads, BLOCK, cfg.hidden_size // cfg.num_attention_heads)
    for _ in range(cfg.num_hidden_layers):
        k = torch.empty(shape, dtype=torch.bfloat16, device=DEV).normal_(0, KV_STD, generator=g)
        v = torch.empty(shape, dtype=torch.bfloat16, device=DEV).normal_(0, KV_STD, generator=g)
        yield k, v


# ------------------------------------------------------------ run
def run(state):
    if state["kind"] == "decode":
        st = state["step"]
        st.set_state(state["ids"], state["pos"])
        st.step()
        return st.logits
    if state["kind"] == "prefill":
        eng, seqs = state["eng"], state["seqs"]
        if len(seqs) == 1:
            logits = eng.prefill(seqs[0], state["ids"])
        else:
            logits = eng.prefill_batch(seqs, state["ids"], use_graph=True)
        return [logits, eng.cache.k[-1], eng.cache.v[-1]]
    for p in state["params"]:
        p.grad = None
    with torch.enable_grad():
        loss = state["model"](state["ids"])
        loss.backward()
    return [loss.detach()] + [p.grad for p in state["params"]]


# ------------------------------------------------------------ QLoRA: a decoder stack as users write them
def rotate_half(x):
    return torch.cat([-x[..., x.shape[-1] // 2:], x[..., :x.shape[-1] // 2]], -1)


def apply_rotary_pos_emb(q, k, cos, sin, unsqueeze_dim=1):
    cos, sin = cos.unsqueeze(unsqueeze_dim), sin.unsqueeze(unsqueeze_dim)
    return q * cos + rotate_half(q) * sin, k * cos + rotate_half(k) * sin


class RMSNorm(nn.Module):
    def __init__(self, w, eps):
        super().__init__()
        self.weight = nn.Parameter(w)
        self.variance_epsilon = eps

    def forward(self, x):
        h = x.float()
        return self.weight * (h * torch.rsqrt(h.pow(2).mean(-1, keepdim=True) + self.variance_epsilon)).to(x.dtype)


def _linear(w):
    m = nn.Linear(w.shape[1], w.shape[0], bias=False, device="meta")
    m.weight = nn.Parameter(w, requires_grad=False)
    return m


class Attention(nn.Module):
    def __init__(self, cfg, w):
        super().__init__()
        self.dim = cfg.hidden_size // cfg.num_attention_heads
        self.q_proj, self.k_proj, self.v_proj, self.o_proj = (_linear(w[n]) for n in "qkvo")

    def forward(self, x, cos, sin):
        from ipex_llm_amd.training.flash_attn import flash_attention
        B, T, _ = x.shape
        q, k, v = (p(x).view(B, T, -1, self.dim).transpose(1, 2) for p in (self.q_proj, self.k_proj, self.v_proj))
        q, k = apply_rotary_pos_emb(q, k, cos, sin)
        return self.o_proj(flash_attention(q, k, v).reshape(B, T, -1))


class GatedMLP(nn.Module):
    def __init__(self, w):
        super().__init__()
        self.gate_proj, self.up_proj, self.down_proj = (_linear(w[n]) for n in ("gate", "up", "down"))
        self.act_fn = nn.SiLU()

    def forward(self, x):
        return self.down_proj(self.act_fn(self.gate_proj(x)) * self.up_proj(x))


class Block(nn.Module):
    def __init__(self, cfg, w):
        super().__init__()
        self.self_attn, self.mlp = Attention(cfg, w), GatedMLP(w)
        self.norm1, self.norm2 = RMSNorm(w["norm1"], cfg.rms_norm_eps), RMSNorm(w["norm2"], cfg.rms_norm_eps)

    def forward(self, x, cos, sin):
        x = x + self.self_attn(self.norm1(x), cos, sin)
        return x + self.mlp(self.norm2(x))


class Decoder(nn.Module):
    def __init__(self, cfg, W):
        super().__init__()
        self.cfg = cfg
        self.embed = nn.Parameter(W.embed())
        self.layers = nn.ModuleList([Block(cfg, W.layer()) for _ in range(W.layers)])
        self.lm_head = _linear(W.normal(cfg.vocab_size, cfg.hidden_size))
        self.norm = RMSNorm(W.norm(), cfg.rms_norm_eps)

    def forward(self, ids):
        from ipex_llm_amd.training.fused_ce import fused_linear_cross_entropy
        x = F.embedding(ids, self.embed)
        cos, sin = _rope(self.cfg, torch.arange(ids.shape[1], device=ids.device), torch.float32)
        cos, sin = cos[None].to(x.dtype), sin[None].to(x.dtype)
        for layer in self.layers:
            x = layer(x, cos, sin)
        return fused_linear_cross_entropy(self.norm(x), self.lm_head.weight, ids)


TARGETS = ["q_proj", "k_proj", "v_proj", "o_proj", "gate_proj", "up_proj", "down_proj"]


def _prepare_train(case, seed):
    from ipex_llm_amd.optimize import optimize_model
    from ipex_llm_amd.training import LoraConfig, get_peft_model
    cfg, r = _config(case), case["rank"]
    W = Weights(cfg, case["layers"], case["qtype"], seed)
    model = Decoder(cfg, W)
    for p in model.parameters():
        p.requires_grad_(False)
    model = optimize_model(model, case["qtype"], modules_to_not_convert=["lm_head"])
    pm = get_peft_model(model, LoraConfig(r=r, lora_alpha=2 * r, target_modules=TARGETS))
    pm.train()
    params = [p for p in pm.parameters() if p.requires_grad]
    for p in params:               # adapters as they are some steps into the training
        p.data.copy_(W.normal(*p.shape, std=0.01))
    return dict(kind="train", model=pm, params=params, ids=_train_ids(case, seed, cfg))


def _train_ids(case, seed, cfg):
    g = torch.Generator().manual_seed(seed + 1)
    return torch.randint(0, cfg.vocab_size, (case["batch"], case["seq"]), generator=g).to(DEV)


# ------------------------------------------------------------ what one pass cannot do without
def work(case):
    cfg = _config(case)
    H, D = cfg.hidden_size, cfg.hidden_size // cfg.num_attention_heads
    L = case.get("layers", cfg.num_hidden_layers)
    layers = L * (2 * H * H + 2 * cfg.num_key_value_heads * D * H + 3 * cfg.intermediate_size * H)
    head = cfg.vocab_size * H
    kv = 4 * cfg.num_key_value_heads * D                        # bytes of a token's key and value
    B, q = case["batch"], BITS[case["qtype"]] / 8
    if case["kind"] == "train":
        T = B * case["seq"]
        adapters = 2 * case["rank"] * L * (9 * H + 2 * cfg.num_key_value_heads * D + 3 * cfg.intermediate_size)
        return {"bytes": layers * q + head * 2 + 2 * adapters,
                "flops": 4 * T * (layers + head) + 3 * adapters * T + L * 3.5 * 2 * H * T * case["seq"]}
    if case["kind"] == "decode":
        keys = B * case["context"] * 0.75
        return {"bytes": (layers + head) * q + L * keys * kv + B * cfg.vocab_size * 2,
                "flops": 2 * B * (layers + head) + L * keys * 4 * H}
    T = B * case["prompt"]
    return {"bytes": (layers + head) * q + L * T * kv,
            "flops": 2 * T * layers + 2 * B * head + L * 2 * H * T * case["prompt"]}


def tolerance(case):
    """a pass is 0.02 off the 64-bit result (16-bit residual stream of 28 to 32 layers; gradients 0.016 to 0.029), and
    two passes whose 32-bit sums come in another order are 0.017 off each other, 0.085 at one value"""
    return {"rel": 0.03, "max": 0.5}


# ------------------------------------------------------------ the same in 64 bits, in plain torch
def _rope(cfg, pos, dtype):
    D = cfg.hidden_size // cfg.num_attention_heads
    inv = 1.0 / (cfg.rope_theta ** (torch.arange(0, D, 2, dtype=torch.float32) / D))
    fr = pos.to(dtype)[:, None] * inv.to(pos.device, dtype)[None]
    fr = torch.cat([fr, fr], -1)
    return fr.cos(), fr.sin()


def _norm(x, w, eps):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * w.double()


def _attend(q, k, v):
    """q [T, heads, D] at the last T of the positions of k / v [L, kv heads, D], causal"""
    T, L, heads, D = q.shape[0], k.shape[0], q.shape[1], q.shape[2]
    kv = k.shape[1]
    hidden = torch.arange(L, device=q.device)[None] > torch.arange(L - T, L, device=q.device)[:, None]
    out = torch.empty_like(q)
    for h in range(kv):
        one = slice(h * heads // kv, (h + 1) * heads // kv)
        s = (q[:, one].transpose(0, 1).reshape(-1, D) @ k[:, h].t()).view(-1, T, L) / math.sqrt(D)
        p = torch.softmax(s.masked_fill_(hidden, float("-inf")), -1)
        out[:, one] = (p.view(-1, L) @ v[:, h]).view(-1, T, D).transpose(0, 1)
    return out


@torch.no_grad()
def exact(case, seed):
    if case["kind"] == "train":
        return _exact_train(case, seed)
    cfg = _config(case)
    nh, nkv, eps, B = cfg.num_attention_heads, cfg.num_key_value_heads, cfg.rms_norm_eps, case["batch"]
    W = Weights(cfg, cfg.num_hidden_layers, case["qtype"], seed)
    D = W.dim
    if case["kind"] == "decode":
        ids, pos = _next_tokens(case, seed, cfg.vocab_size)
        cached = _cached(case, seed, cfg)
    else:
        ids, cached = _tokens(case, seed, cfg.vocab_size).reshape(-1), None
        pos = torch.arange(case["prompt"]).repeat(B)
    cos, sin = (t[:, None] for t in _rope(cfg, pos.to(DEV), torch.float64))
    x = W.embed()[ids.to(DEV)].double()
    T = x.shape[0] // B
    for _ in range(cfg.num_hidden_layers):
        w = W.layer()
        y = _norm(x, w["norm1"], eps) @ torch.cat([w["q"], w["k"], w["v"]]).double().t()
        if "bias" in w:
            y += w["bias"].double()
        qh, kh, vh = y.view(-1, nh + 2 * nkv, D).split([nh, nkv, nkv], 1)
        qh, kh = (t * cos + rotate_half(t) * sin for t in (qh, kh))
        old, outs = (next(cached) if cached is not None else None), []
        for b in range(B):
            at = slice(b * T, (b + 1) * T)
            kb, vb = kh[at], vh[at]
            if old is not None:
                n = int(pos[b])
                past = [t.view(B, -1, nkv, BLOCK, D)[b].transpose(1, 2).reshape(-1, nkv, D)[:n].double() for t in old]
                kb, vb = torch.cat([past[0], kb]), torch.cat([past[1], vb])
            outs.append(_attend(qh[at], kb, vb))
        x = x + torch.cat(outs).reshape(x.shape[0], -1) @ w["o"].double().t()
        h = _norm(x, w["norm2"], eps)
        x = x + (F.silu(h @ w["gate"].double().t()) * (h @ w["up"].double().t())) @ w["down"].double().t()
        del w
    head = W.grid(cfg.vocab_size, cfg.hidden_size)
    x = _norm(x[T - 1::T], W.norm(), eps)
    logits = torch.cat([x @ w.double().t() for w in head.split(32768)], -1)
    return logits if case["kind"] == "decode" else [logits, None, None]


def _exact_train(case, seed):
    cfg, r = _config(case), case["rank"]
    W = Weights(cfg, case["layers"], case["qtype"], seed)
    model = Decoder(cfg, W)
    weights = {n: p.detach() for n, p in model.named_parameters()}
    names = [n for n, m in model.named_modules() if isinstance(m, nn.Linear) and n != "lm_head"]
    del model
    ab = {}
    for n in names:
        out, k = weights[n + ".weight"].shape
        ab[n] = [W.normal(r, k, std=0.01).double().requires_grad_(), W.normal(out, r, std=0.01).double().requires_grad_()]
    ids = _train_ids(case, seed, cfg)
    B, T = ids.shape
    nh, nkv, D, eps = cfg.num_attention_heads, cfg.num_key_value_heads, W.dim, cfg.rms_norm_eps
    cos, sin = (t[None, None] for t in _rope(cfg, torch.arange(T, device=DEV), torch.float64))
    hidden = torch.ones(T, T, dtype=torch.bool, device=DEV).triu(1)

    def linear(x, n):
        a, b = ab[n]
        return x @ weights[n + ".weight"].double().t() + 2 * ((x @ a.t()) @ b.t())

    def block(x, n):
        h = _norm(x, weights[n + ".norm1.weight"], eps)
        qh, kh, vh = (linear(h, f"{n}.self_attn.{c}_proj").view(B, T, -1, D).transpose(1, 2) for c in "qkv")
        qh, kh = (t * cos + rotate_half(t) * sin for t in (qh, kh))
        s = (qh.reshape(B, nkv, nh // nkv, T, D) @ kh[:, :, None].transpose(-1, -2)) / math.sqrt(D)
        o = torch.softmax(s.masked_fill(hidden, float("-inf")), -1) @ vh[:, :, None]
        x = x + linear(o.reshape(B, nh, T, D).transpose(1, 2).reshape(B, T, -1), f"{n}.self_attn.o_proj")
        h = _norm(x, weights[n + ".norm2.weight"], eps)
        h = F.silu(linear(h, f"{n}.mlp.gate_proj")) * linear(h, f"{n}.mlp.up_proj")
        return x + linear(h, f"{n}.mlp.down_proj")

    with torch.enable_grad():
        x = weights["embed"][ids].double()
        for i in range(case["layers"]):
            x = torch.utils.checkpoint.checkpoint(block, x, f"layers.{i}", use_reentrant=False)
        h = _norm(x, weights["norm.weight"], eps)[:, :-1].reshape(-1, cfg.hidden_size)
        want = ids[:, 1:].reshape(-1)
        # head and loss some rows at a time, their gradient carried on by hand
        hd, loss, n = h.detach().requires_grad_(), 0.0, want.numel()
        head = weights["lm_head.weight"].double()
        for at in range(0, n, 1024):
            part = F.cross_entropy(hd[at:at + 1024] @ head.t(), want[at:at + 1024], reduction="sum") / n
            part.backward()
            loss = loss + part.detach()
        h.backward(hd.grad)
    return [loss] + [t.grad for n in names for t in ab[n]]
