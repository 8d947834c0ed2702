"""Prefill-size (M > 64) low-bit GEMM dispatch.

Three paths: the skinny kernel (``csrc/hip/lowbit_skinny.cuh``: the decode
kernel for 17 rows and up, weights streamed once, codes raw in the MFMA) while
its row blocks fit one round of the chip; the MFMA kernel with in-register
dequant (``csrc/hip/gemm.hip``: f16 MFMA, weights decoded straight from the
tiled blob, never materialised) for the wide gate/up pairs above that; and
dequantize to a transient dense weight + GEMM.  Measured on MI355X (Llama-3-8B,
sym_int4, graph replays over weights that no cache holds), skinny against the
better of the other two: M = 96 qkv 19 / 38 us, o 15 / 38, down 25 / 75,
gate_up 41 / 58; M = 300 qkv 28 / 44, o 27 / 37, down 71 / 93, gate_up
119 / 112; M = 512 o 28 / 38, down 86 / 104, qkv (two rounds) 52 / 48.
``ILLM_GEMM_LIB=1`` / ``ILLM_GEMM_FUSED=1`` force either other path (A/B runs).
"""
from __future__ import annotations

import contextlib
import os
import statistics
import weakref
from typing import Dict

import torch
import torch.nn.functional as F

_USE_LIB = os.environ.get("ILLM_GEMM_LIB", "0") == "1"
_USE_FUSED = os.environ.get("ILLM_GEMM_FUSED", "0") == "1"
FUSED_MAX_M = 128          # fused kernel for every shape up to here (K <= FUSED_LONG_K)
FUSED_LONG_K = 8192        # deeper K (down projections): library path from M > 64
FUSED_QKV_MAX_M = 256      # N >= 6144 (fused qkv) up to here
FUSED_WIDE_MAX_M = 384     # N >= FUSED_WIDE_N (gate/up pairs) up to here
FUSED_WIDE_N = 12288


ROWS_MAX_M = 512           # skinny kernel up to here (from 512 rows on the dense paths are tiled for them)


def rows_fit(M: int, n: int, fmt: int, glu: bool = False, k: int = 0) -> bool:
    """The skinny kernel's 64-row x 128-column blocks fit one round of the 256
    CUs (a second round costs what the first did, and the compute-bound paths
    are then ahead); formats with block minima, whose sums take a third more,
    up to 5 / 8 of that and 320 rows (asym_int5 [2048, 2048], 300 rows 17.5 /
    18.3 us, 384 rows 17.7 / 19.3), asym_int5 up to a half ([4096, 8192] 320
    rows 62 / 57).  Gate/up pairs by the rows alone -- a column shard of a
    tensor-parallel model takes the kernel that the whole pair takes --: up to 96
    rows (Llama-3-8B sym_int4, this / the fused kernel: M = 65 42 / 58 us, 96
    41 / 58; two and more rounds would take 128 rows there, 49 / 58, not in
    [37888, 3584], 64 / 63), and 8-bit floats, whose codes have no offset, up to
    512 (fp8_e5m2 [37888, 3584] M = 128 62 / 73, 300 118 / 128, 512 192 / 196;
    e4m3 [28672, 4096] 50 / 58, 105 / 122, 152 / 168; not of K up to 1024,
    [14336, 1024] M = 420 44 / 34).  Nor pairs of over three rounds where a round
    is short or has minima in integer bytes ([151936, 1024] sym_int4 80 / 70,
    fp4 77 / 62; [57344, 8192] asym_int5 219 / 209, sym_int4 158 / 185)."""
    if _USE_LIB or _USE_FUSED or M > ROWS_MAX_M:
        return False
    from ..quantize import qtypes as Q
    if glu:
        if fmt in (Q.FMT_FP8E4, Q.FMT_FP8E5, Q.FMT_FP6) and not 0 < k <= 1024:
            return True
        return M <= 96 and not (n > 49152 and (0 < k <= 1024 or fmt == Q.FMT_ASYM_INT5))
    blocks = (n + 127) // 128 * ((M + 63) // 64)
    if fmt in (Q.FMT_ASYM_INT4, Q.FMT_ASYM_INT5):
        return blocks <= (160 if fmt == Q.FMT_ASYM_INT4 else 128) and M <= 320
    return blocks <= 256


def rows_take(dtype, M: int, n: int, k: int, fmt: int, glu: bool = False) -> bool:
    """... and it loses no bit against the path it replaces.  A gate/up pair of
    the fused kernel with a table weight under bf16 stays there: the finer table
    (:func:`rows_fine`) is the longer one over two rounds (nf4 [28672, 4096], 80
    rows 65 / 60 us; [8192, 1024] 10 / 17, but by the rows alone, as above)."""
    if M < 1 or dtype not in (torch.bfloat16, torch.float16) or not rows_fit(M, n, fmt, glu, k):
        return False
    return not (rows_fine(dtype, M, n, k, fmt) and (glu or M <= 64))


def rows_fine(dtype, M: int, n: int, k: int, fmt: int) -> bool:
    """The skinny kernel's 16-bit table is in the type of x: a weight error of
    1.4e-3 in bf16.  A dense bf16 weight has 1.7e-3, but the fused kernel's f16
    table 1.8e-4: its products take a table of bf16 pairs (1e-5), which costs up
    to a third (nf4 [6144, 4096], us, one / pairs / fused kernel: 80 rows 20.5 /
    24.3 / 42.6, 256 rows 29 / 38 / 45; [8192, 8192] 80 rows 31 / 40 / 79)."""
    from ..quantize import qtypes as Q
    return dtype == torch.bfloat16 and fmt in (Q.FMT_NF4, Q.FMT_NF3) and use_fused(M, n, k)


def use_rows(x, M: int, n: int, k: int, fmt: int, glu: bool = False) -> bool:
    # the op has no derivative, the library product over a dense weight has
    derived = (x.requires_grad and torch.is_grad_enabled()) or torch.autograd.forward_ad._current_level >= 0
    return x.is_cuda and not derived and rows_take(x.dtype, M, n, k, fmt, glu)


def use_fused(M: int, n: int, k: int = 0) -> bool:
    if _USE_LIB:
        return False
    if _USE_FUSED:
        return True
    if k > FUSED_LONG_K:
        return M <= 64
    if n >= FUSED_WIDE_N:
        return M <= FUSED_WIDE_MAX_M
    if n >= 6144:
        return M <= FUSED_QKV_MAX_M
    return M <= FUSED_MAX_M


def wants_dense(dtype, M: int, n: int, k: int, fmt: int, glu: bool = False) -> bool:
    """the product expands its weight: what ``lowbit_gemm`` and ``lowbit_gemm_glu``
    ask, in their order (a pair that no pair kernel takes is a plain product)"""
    if rows_take(dtype, M, n, k, fmt, glu):
        return False
    if g8d_takes(dtype, M, n, k, glu):
        return True
    if use_fused(M, n, k):
        return False
    return not glu or wants_dense(dtype, M, n, k, fmt)


# ---- dense-weight prefetch for the library path ---------------------------
# The library path's dequantize is memory-bound and the GEMM it feeds is
# compute-bound: the decoder asks for the NEXT layer's dense weights while
# the current layer computes, and they are written on a side HIP stream, so
# the dequant traffic overlaps the MFMA work instead of sitting between the
# GEMMs.  At most one layer's weights are held ahead (consumed entries are
# dropped).  Opt-in (ILLM_GEMM_PREFETCH=1): measured on MI355X (Llama-3-8B,
# 1024-token prompts) the overlapped dequant contends with the GEMMs for HBM
# and CUs -- first token B=1 21.1 -> 22.0 ms, B=8 104.3 -> 103.3 ms.
_PREFETCH = os.environ.get("ILLM_GEMM_PREFETCH", "0") == "1"
_ready = {}                 # (blob ptr, n, k, dtype) -> (dense weight, event)
_side = {}                  # device index -> side stream


def _key(blob, n, k, dtype):
    return (blob.data_ptr(), n, k, dtype)


def prefetch_dense(items, M: int, dtype) -> None:
    """Dequantize ``items`` = [(blob, fmt, n, k, glu)] on a side stream for an
    upcoming library-path GEMM with M rows (no-op for the shapes that the
    skinny or the fused kernel takes, during graph capture, or when disabled)."""
    if not _PREFETCH or not items or torch.cuda.is_current_stream_capturing():
        return
    ops = torch.ops.ipex_llm_amd
    for blob, fmt, n, k, glu in items:
        if not blob.is_cuda or not wants_dense(dtype, M, n, k, fmt, glu):
            continue
        key = _key(blob, n, k, dtype)
        if key in _ready:
            continue
        dev = blob.device.index
        st = _side.get(dev)
        if st is None:
            st = _side[dev] = torch.cuda.Stream(device=blob.device)
        with torch.cuda.stream(st):
            w = ops.dequantize_device(blob, fmt, n, k, dtype)
            ev = torch.cuda.Event()
            ev.record(st)
        _ready[key] = (w, ev)


# ---- resident dense shadow of the low-bit weights for prefill -------------
# Decode streams the low-bit blob (bandwidth-bound); prefill at M >= 512 is
# compute-bound and runs the library GEMM on a dequantized copy that the path
# above re-creates on every call (2 B/weight written and re-read: ~20 % of a
# 1024-token prefill GEMM).  With 288 GB of HBM3E per MI355X the dequantized
# copy can simply stay resident: ILLM_PREFILL_DENSE_GB=<budget> keeps up to
# that many GB of bf16/f16 shadows (first use dequantizes, later prefills
# reuse it; numerics identical to the dequantize-per-call path).  Default 0:
# nothing kept (the low-bit footprint only).
_DENSE_BUDGET = float(os.environ.get("ILLM_PREFILL_DENSE_GB", "0")) * 2 ** 30
_dense_bytes = [0]           # bytes charged to the budget by every resident shadow (incl. training/lora.py's)


class ChargedCache(dict):
    """key -> (weakref to blob, shadow, charged bytes): removing an entry (pop,
    del, clear, the blob's weakref callback) refunds its bytes to the budget"""

    def pop(self, key, *default):
        ent = super().pop(key, None)
        if ent is None:
            return default[0] if default else None
        _dense_bytes[0] -= ent[2]
        # entries of other caches that view this entry's storage (charged 0) go too:
        # a surviving view would keep the bytes alive after their refund
        for c, k in self.__dict__.get("_links", {}).pop(key, ()):
            c.pop(k)
        return ent

    def link(self, key, other: "ChargedCache", okey):
        """drop ``other[okey]`` (a view of this entry's shadow) with ``self[key]``"""
        self.__dict__.setdefault("_links", {}).setdefault(key, []).append((other, okey))

    def __delitem__(self, key):
        self.pop(key)

    def clear(self):
        for k in list(self.keys()):
            self.pop(k)

    def _pop_if(self, key, ref):
        ent = self.get(key)
        if ent is not None and ent[0] is ref:      # a newer entry under a reused address stays
            self.pop(key)

    def put(self, key, blob, w, charged: int):
        self.pop(key)
        super().__setitem__(key, (weakref.ref(blob, lambda r, key=key, c=self: c._pop_if(key, r)), w, charged))
        _dense_bytes[0] += charged


_dense_cache = ChargedCache()  # (blob ptr, version, n, k, dtype) -> (weakref to blob, dense weight, bytes)


def dense_fits(nbytes: int) -> bool:
    """another ``nbytes`` of resident shadow stays within the budget"""
    return _DENSE_BUDGET > 0 and _dense_bytes[0] + nbytes <= _DENSE_BUDGET


# a prefill graph being captured records the addresses of the shadows it reads:
# they are pinned in the graph's own entry (Engine._pf_graphs), so dropping a
# cache entry (budget change, dense_cache_clear) can never free memory a
# captured graph still reads
_capture_pins = None


@contextlib.contextmanager
def pin_dense_shadows():
    global _capture_pins
    prev, _capture_pins = _capture_pins, []
    try:
        yield _capture_pins
    finally:
        _capture_pins = prev


def set_dense_budget(gb: float) -> None:
    """budget (GiB) of dequantized weights kept resident by ``_dense_weight``
    (frozen low-bit weights: the cache never goes stale); 0 disables"""
    global _DENSE_BUDGET
    _DENSE_BUDGET = float(gb) * 2 ** 30
    if _DENSE_BUDGET <= 0:
        dense_cache_clear()


def dense_cache_clear() -> None:
    _dense_cache.clear()


def auto_dense_budget(device, cap_gb: float = float("inf")) -> float:
    """Inference default for the prefill shadow (engine construction): an
    explicit ILLM_PREFILL_DENSE_GB wins; otherwise 0 -- the model keeps its
    low-bit footprint only and prefill dequantizes each weight once per GEMM
    into a transient buffer for the dense 8-phase kernel (``use_g8d``).  A
    resident shadow (ILLM_PREFILL_DENSE_GB=48 on MI355X: a Llama-3-8B INT4
    model adds 15 GB next to its 4.5 GB) saves that ~3-4 % dequant pass;
    ``cap_gb`` bounds an explicit request.  Returns the budget in GiB."""
    env = os.environ.get("ILLM_PREFILL_DENSE_GB")
    gb = min(float(env), cap_gb) if env is not None else 0.0
    if gb * 2 ** 30 > _DENSE_BUDGET:
        set_dense_budget(gb)
    return gb


def _dense_drop(key):
    _dense_cache.pop(key, None)


def _dense_weight(blob, fmt, n, k, dtype):
    if _DENSE_BUDGET > 0:
        # keyed by address, validated by identity: an entry lives exactly as
        # long as its blob (weakref callback), so a later model whose blob
        # reuses the address never sees another model's weights
        key = (blob.data_ptr(), blob._version, n, k, dtype)
        ent = _dense_cache.get(key)
        if ent is not None:
            if ent[0]() is blob:
                if _capture_pins is not None and torch.cuda.is_current_stream_capturing():
                    _capture_pins.append(ent[1])
                return ent[1]
            _dense_drop(key)
        w = torch.ops.ipex_llm_amd.dequantize_device(blob, fmt, n, k, dtype)
        if torch.cuda.is_current_stream_capturing():
            return w                # captured: a transient of the graph's pool, never cached
        nb = w.numel() * w.element_size()
        if dense_fits(nb):
            _dense_cache.put(key, blob, w, nb)
        return w
    hit = _ready.pop(_key(blob, n, k, dtype), None) if _ready else None
    if hit is None:
        return torch.ops.ipex_llm_amd.dequantize_device(blob, fmt, n, k, dtype)
    w, ev = hit
    cur = torch.cuda.current_stream(blob.device)
    cur.wait_event(ev)
    w.record_stream(cur)           # allocated on the side stream, used (and freed) here
    return w


def drop_prefetched() -> None:
    """Release prefetched weights nobody consumed (e.g. an aborted forward)."""
    _ready.clear()


# ---- the 8-phase 256 x 256 GEMM (csrc/hip/gemm_8p.hip): bf16 MFMA, weights
# decoded to bf16 in LDS just in time (bit-identical to dequantize-to-bf16 +
# GEMM), LDS-DMA activations, counted-vmcnt pipeline, staggered wave-rows.
# sym_int4 and the nf4 / nf3 LUT formats; bf16 activations; from G8_MIN_M rows
# (ILLM_GEMM_8P=0 disables it).
_G8 = os.environ.get("ILLM_GEMM_8P", "0") == "1"     # opt-in: 0.6-0.7x dequant + hipBLASLt so far (profiles/gemm8p_sweep_r4.jsonl)
G8_MIN_M = int(os.environ.get("ILLM_GEMM_8P_MIN_M", "1024"))
_G8_FMTS = None


def _g8_fmts():
    global _G8_FMTS
    if _G8_FMTS is None:
        from ..quantize import get_format
        _G8_FMTS = {get_format(q).fmt for q in ("sym_int4", "nf4", "nf3")}
    return _G8_FMTS


def use_g8(x, M: int, n: int, k: int, fmt: int, glu: bool = False) -> bool:
    return (_G8 and not _USE_LIB and not _USE_FUSED and x.is_cuda and x.dtype == torch.bfloat16 and M >= G8_MIN_M
            and k % 128 == 0 and (not glu or n % 32 == 0) and fmt in _g8_fmts() and _DENSE_BUDGET <= 0
            and hasattr(torch.ops.ipex_llm_amd, "gemm8p_lowbit"))


# ---- default prefill path: stream-dequantize + the dense 8-phase GEMM -------
# The in-LDS-dequant kernel above decodes every weight tile once per 256-row
# M block (32 times at M = 8192); on gfx950 that decode (~3.5 VALU per weight)
# competes with the MFMAs for the SIMD's vector issue (an MFMA holds it 8 of
# its 16 cycles) and the kernel runs at ~0.67x of a dense GEMM
# (profiles/g8_sched_sweep_r5.jsonl).  Decoding each weight ONCE into a
# transient bf16 copy (dequantize_device, HBM-bound: ~3-4 % of the GEMM) and
# running the dense 8-phase kernel (gemm_8p.hip: LDS-DMA, counted vmcnt,
# split-K for grids smaller than the chip, GLU in the epilogue) keeps the
# low-bit footprint -- no resident shadow -- and no library GEMM.
# ILLM_GEMM_G8D=0 falls back to dequantize + hipBLASLt (A/B).
_G8D = os.environ.get("ILLM_GEMM_G8D", "1") == "1"
G8D_MIN_M = int(os.environ.get("ILLM_GEMM_G8D_MIN_M", "512"))


def g8d_takes(dtype, M: int, n: int, k: int, glu: bool = False) -> bool:
    return (_G8D and not _USE_LIB and not _USE_FUSED and dtype == torch.bfloat16
            and M >= G8D_MIN_M and k % 64 == 0 and (not glu or n % 32 == 0)
            and hasattr(torch.ops.ipex_llm_amd, "gemm_bf16"))


def use_g8d(x, M: int, n: int, k: int, glu: bool = False) -> bool:
    return x.is_cuda and g8d_takes(x.dtype, M, n, k, glu)


# ---- measured dispatch: dense 8-phase kernel vs the library GEMM -----------
# Over the same transient bf16 weight, the 8-phase kernel reaches 0.8-0.9x
# hipBLASLt at M = 8192 and 0.5-0.8x at M = 1024 (profiles/g8d_slab_splitk_sweep_r5.jsonl);
# end to end the library path took the Llama-3-8B first token from 98.9 to 90.3 ms
# at B = 8 x 1024 and 19.8 to 18.5 ms at B = 1 (profiles/prefill_lib_ab_r6.jsonl).
# Each (M, N, K, GLU) shape times both once, outside graph capture (the engine's
# eager warm-up precedes every prefill capture), and keeps the faster; a shape first
# seen under capture takes the 8-phase kernel.  ILLM_GEMM_AUTOTUNE=0: always 8-phase.
_AUTOTUNE = os.environ.get("ILLM_GEMM_AUTOTUNE", "1") == "1"
# A later candidate is taken from this share of an earlier one's time on.  The candidates round differently, so where two
# are as fast -- a 1024-row [4096, 14336] product, 8-phase 137.7 to 139.1 us, library 140.0 to 141.0 -- the logits of a
# prompt were now one's and now the other's, 0.02 apart, by the noise of the process that timed them.  The line is where
# the larger products leave a gap, on each side of 1024 rows.  Library / 8-phase, medians, over processes and cards: 1024 rows
# [28672, 4096] pairs 0.996 to 1.09 and [4096, 14336] 0.992 to 1.03, qkv and o 0.71 to 0.78; 8192 rows [28672, 4096] pairs
# 0.945 to 0.967, 4096 rows 0.923 to 0.976, [3584, 18944] 0.933 to 0.956, the others 0.80 to 0.87.  (With one line for all, at
# 0.97 or 0.98, one of the two was within 2 % of it, the difference of two cards.)
_AHEAD_FEW, _AHEAD_MANY = 0.95, 1.0        # up to 1024 rows, above


def _ahead(M: int) -> float:
    return _AHEAD_FEW if M <= 1024 else _AHEAD_MANY


_CHOICE: Dict[tuple, str] = {}


def _rounds(fns, rounds: int, reps: int = 3):
    """GPU time of each candidate in each of the rounds, the candidates in turn"""
    t0, t1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    out = []
    for _ in range(rounds):
        out.append([])
        for fn in fns:
            torch.cuda._sleep(200000)
            t0.record()
            for _ in range(reps):
                fn()
            t1.record()
            t1.synchronize()
            out[-1].append(t0.elapsed_time(t1) / reps)
    return out


def _time_ms(fns):
    """GPU time of each candidate, the best over three rounds in turn.  A single round is off by
    more than the candidates differ, since the library's first calls of a process are in it:
    at [6144, 4096] and 1024 rows it read 82 (8-phase) and 136 us (library) for what are 82
    and 65 us, in each of five processes, and a 1024-token Llama-3-8B prompt took 18.4 to
    18.7 ms instead of 18.0 (18.5 in the one process of five whose gate/up pair, 249 to 271
    against 268 us, fell to the slower side).  The calls are queued behind 90 us of waiting
    on the GPU: without it the gaps between launches, which graph replays do not have,
    decide small products ([2048, 2048] pairs of 512 rows, 34 / 25 us, read 36 / 34).
    Once per shape and process: 10 calls of each candidate, and 18 more of candidates that are
    within 10 % of another, whose medians over all rounds are then taken (the best
    of three rounds of the 8192-row [28672, 4096] pair read 0.940 to 0.977)"""
    for fn in fns:
        fn()
    times = _rounds(fns, 3)
    best = [min(t) for t in zip(*times)]
    if any(abs(t / best[i] - 1) < 0.1 for i in range(len(best)) for t in best[i + 1:]):
        times += _rounds(fns, 6)
        best = [statistics.median(t) for t in zip(*times)]
    return best


def _mbucket(M: int) -> int:
    """rows rounded up to a power of two: serving sees every prompt length, and one
    timing per bucket keeps the table (and the warm-up cost) bounded"""
    return 1 << max(0, int(M) - 1).bit_length()


def _pick(key: tuple, g8d_fn, lib_fn, *more) -> str:
    """'g8d' | 'lib' | 'lib1' ... (the extra candidates ``more``, in order);
    key = (M, N, K, kind, act), M bucketed"""
    key = (_mbucket(key[0]),) + tuple(key[1:])
    c = _CHOICE.get(key)
    if c is None:
        if not _AUTOTUNE or torch.cuda.is_current_stream_capturing():
            return "g8d"
        names = ["g8d", "lib"] + [f"lib{i + 1}" for i in range(len(more))]
        times = _time_ms((g8d_fn, lib_fn) + more)
        ahead, best = _ahead(key[0]), 0
        for i, t in enumerate(times):
            if t < ahead * times[best]:
                best = i
        c = _CHOICE[key] = names[best]
        if os.environ.get("ILLM_GEMM_AUTOTUNE_LOG"):
            print(f"[gemm] M={key[0]} N={key[1]} K={key[2]} glu={key[3]}: "
                  + ", ".join(f"{n} {t * 1e3:.1f} us" for n, t in zip(names, times)) + f" -> {c}", flush=True)
    return c


def gemm_choices() -> Dict[tuple, str]:
    """the measured per-shape choices so far: (M, N, K, glu, act) -> 'g8d' | 'lib'"""
    return dict(_CHOICE)


def lowbit_gemm(x, blob, fmt, n, k, bias=None):
    ops = torch.ops.ipex_llm_amd
    M = x.numel() // k
    bf16_bias = bias is None or bias.dtype == torch.bfloat16
    if use_rows(x, M, n, k, fmt) and (bias is None or bias.dtype == x.dtype):
        return ops.gemm_rows(x, blob, fmt, n, k, bias, False, 0, rows_fine(x.dtype, M, n, k, fmt))
    if use_g8(x, M, n, k, fmt) and bf16_bias:
        return ops.gemm8p_lowbit(x, blob, fmt, n, k, bias)
    if use_g8d(x, M, n, k) and bf16_bias:
        # candidates timed with their weight preparation: the 8-phase kernel and
        # the library over the transient bf16 weight.  (The in-LDS low-bit
        # 8-phase kernel, no transient weight, lost every Llama-3-8B prefill shape
        # as a third candidate: 0.55-0.85x, profiles/prefill_choices_b{1,8}_r6.txt.)
        def dw():
            return _dense_weight(blob, fmt, n, k, x.dtype)
        c = _pick((M, n, k, False, 0), lambda: ops.gemm_bf16(x, dw(), bias), lambda: F.linear(x, dw(), bias))
        return F.linear(x, dw(), bias) if c == "lib" else ops.gemm_bf16(x, dw(), bias)
    if use_fused(M, n, k) and hasattr(ops, "gemm"):
        return ops.gemm(x, blob, fmt, n, k, bias)
    w = _dense_weight(blob, fmt, n, k, x.dtype)
    return F.linear(x, w, bias)


def lowbit_slabs(x, blob, fmt, n, k, least=1):
    """x @ W^T of more rows than the decode kernels take as the f32 slabs [S, M, n]
    of a split K for :func:`add_rms_norm` to sum -- it rounds the sum as the pass
    over the slabs that this saves does, so with the same bits --, or None where
    the skinny kernel makes fewer than ``least`` or :func:`lowbit_gemm` takes a dense
    product that it does not split.  Product and norm, us, of slabs / of the 16-bit
    result: fp8_e5m2 [3584, 18944] of 300 rows, three slabs, 70.3 / 73.9; a product in
    one piece has no pass to save, and its slab is twice the bytes: [3584, 3584] of 300
    rows 24.9 / 24.0, sym_int4 [4096, 14336] of 512 rows 86.3 / 83.8.  Pass and norm /
    norm alone of the dense [4096, 14336] of 1024 rows 22.5 / 16.2."""
    ops = torch.ops.ipex_llm_amd
    M = x.numel() // k
    if torch.is_grad_enabled() and x.requires_grad:
        return None
    if use_rows(x, M, n, k, fmt):
        fine = rows_fine(x.dtype, M, n, k, fmt)
        if least > 1 and ops.gemv_slabs(M, n, k, fmt, x.dtype == torch.bfloat16, 0, fine) < least:
            return None
        return ops.gemm_rows_slabs(x, blob, fmt, n, k, fine)
    if use_g8(x, M, n, k, fmt) or not use_g8d(x, M, n, k) or ops.gemm_bf16_split(M, n, k) < 2:
        return None

    def dw():
        return _dense_weight(blob, fmt, n, k, x.dtype)
    if _pick((M, n, k, False, 0), lambda: ops.gemm_bf16(x, dw()), lambda: F.linear(x, dw())) == "lib":
        return None
    return ops.gemm_bf16_slabs(x, dw())


def lowbit_gemm_glu(x, blob, fmt, n, k, act: int = 0):
    """act(x @ Wg^T) * (x @ Wu^T) for a tile-interleaved gate/up weight at
    prefill M: the fused kernel applies the activation in its epilogue (no
    [M, 2I] round trip, no elementwise launches)."""
    ops = torch.ops.ipex_llm_amd
    M = x.numel() // k
    if use_rows(x, M, n, k, fmt, glu=True):
        return ops.gemm_rows(x, blob, fmt, n, k, None, True, act)
    if use_g8(x, M, n, k, fmt, glu=True):
        return ops.gemm8p_lowbit(x, blob, fmt, n, k, None, False, True, act)
    if use_g8d(x, M, n, k, glu=True) and act in (0, 1):
        from .api import glu

        def dw():
            return _dense_weight(blob, fmt, n, k, x.dtype)

        def lib():
            return glu(F.linear(x, dw()), act, tile=16)
        c = _pick((M, n, k, True, act), lambda: ops.gemm_bf16(x, dw(), None, False, 0, True, act), lib)
        return lib() if c == "lib" else ops.gemm_bf16(x, dw(), None, False, 0, True, act)
    if use_fused(M, n, k) and hasattr(ops, "gemm_glu"):
        return ops.gemm_glu(x, blob, fmt, n, k, act)
    from .api import glu
    return glu(lowbit_gemm(x, blob, fmt, n, k), act, tile=16)
