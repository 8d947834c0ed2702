"""Decode attention whose workgroups stream a pair's keys (attn_dec_v4.cuh) against float64: sequence ends at the edges of a
wave's 32 keys and of 4- and 8-wave tiles, waves without keys, one workgroup a pair and several, more than 64 tiles a wave,
blocks that are no power of two, windows, softcap and ALiBi, q from memory and pre-rotated with the new token appended."""
import pytest
import torch

import ipex_llm_amd.ops as ops

pytestmark = pytest.mark.gpu
EDGES = [1, 31, 32, 33, 127, 128, 129, 255, 256, 257, 511, 512, 513]


def _reference(L, kc, vc, bt, q, scale, softcap, window, alibi):
    """float64 results and the weighted sum of the values' magnitudes"""
    Hkv, Hq = kc.shape[1], q.shape[2]
    refs, mags = [], []
    for b, n in enumerate(L):
        k, v = (c[bt[b].long()].transpose(1, 2).reshape(-1, Hkv, c.shape[-1])[:n].double() for c in (kc, vc))
        x = q[b].double().view(q.shape[1], Hkv, Hq // Hkv, -1)
        s = torch.stack([x[:, h] @ k[:, h].t() for h in range(Hkv)], 1).reshape(q.shape[1], Hq, n) * scale
        s = softcap * torch.tanh(s / softcap) if softcap else s
        key, pos = torch.arange(n, device=q.device), torch.arange(q.shape[1], device=q.device)[:, None, None] + n - q.shape[1]
        if alibi is not None:
            s = s + alibi.double()[None, :, None] * key
        ok = (key <= pos) & ((key > pos - window) if window else True)
        p = s.masked_fill(~ok, float("-inf")).softmax(-1).view(q.shape[1], Hkv, Hq // Hkv, n)
        refs.append(torch.stack([p[:, h] @ v[:, h] for h in range(Hkv)], 1).reshape(q.shape[1], Hq, -1))
        mags.append(torch.stack([p[:, h] @ v[:, h].abs() for h in range(Hkv)], 1).reshape(q.shape[1], Hq, -1))
    return refs, mags


def _setup(dev, L, cap, Hkv, bs, dtype):
    torch.manual_seed(len(L) * cap + bs)
    nb = -(-cap // bs)
    kc, vc = (torch.randn(nb * len(L), Hkv, bs, 128, device=dev).to(dtype) for _ in range(2))
    bt = torch.randperm(nb * len(L), device=dev).int().view(len(L), nb).contiguous()
    return kc, vc, bt, torch.tensor(L, dtype=torch.int32, device=dev), -(-cap // 64)


CASES = [  # lengths, keys of the grid, kv heads, group, block, (waves, workgroups)
    ([EDGES[i % 13] for i in range(17)], 640, 8, 4, 64, [8, 1]),
    ([EDGES[i % 13] for i in range(40)], 640, 8, 1, 64, [4, 1]),
    ([1, 32, 129, 191, 192] * 2, 192, 8, 4, 192, [4, 1]),
    ([511, 33, 1] * 3, 512, 2, 16, 128, [8, 1]),
    ([1024, 895, 129, 127, 128, 1, 640, 960], 1088, 8, 7, 64, [4, 8]),
    ([4100, 2047, 33], 4224, 8, 4, 192, [4, 16]),
    ([17000, 16384, 1] + [65] * 14, 17024, 8, 2, 64, [4, 17]),     # 8 tiles in a row a workgroup, most without keys
    ([1344, 1025, 1024, 1023, 129, 1, 33, 64] * 5, 1344, 8, 4, 64, [4, 2]),
    ([2624, 2048, 2049, 1] + [200] * 14, 2688, 8, 7, 192, [4, 3]),
    ([25600, 1, 33, 128, 129], 25600, 27, 1, 64, [4, 3]),          # 67 tiles a wave
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("L,cap,Hkv,G,bs,plan", CASES)
@pytest.mark.parametrize("softcap,window,slopes", [(0.0, 0, False), (30.0, 100, True)])
def test_q_from_memory(cuda, L, cap, Hkv, G, bs, plan, softcap, window, slopes, dtype):
    kc, vc, bt, sl, ns = _setup(cuda, L, cap, Hkv, bs, dtype)
    assert torch.ops.ipex_llm_amd.attn_decode_plan(len(L), Hkv, ns) == plan
    for Tq in (1, 2) if G <= 8 and min(L) > 1 else (1,):
        q = torch.randn(len(L), Tq, Hkv * G, 128, device=cuda).to(dtype)
        alibi = torch.linspace(0.001, 0.05, Hkv * G, device=cuda) if slopes else None
        got = ops.attn_decode(q, kc, vc, bt, sl, ns, 128 ** -0.5, softcap, window, alibi=alibi).view_as(q)
        u = torch.finfo(dtype).eps / 2
        for b, (ref, mag) in enumerate(zip(*_reference(L, kc, vc, bt, q, 128 ** -0.5, softcap, window, alibi))):
            # p and the result are each rounded by at most u; 5 % on top for the f32 scores, exponentials and sums
            assert ((got[b].double() - ref).abs() <= 2.1 * u * mag + 1e-30).all(), (b, L[b])
    ops.check_kernel_errors(cuda)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("L,cap,Hkv,G,bs,plan", CASES)
@pytest.mark.parametrize("window", [0, 300])
def test_pre_rotated(cuda, L, cap, Hkv, G, bs, plan, window, dtype):
    kc, vc, bt, sl, ns = _setup(cuda, L, cap, Hkv, bs, dtype)
    B, Hq, D = len(L), Hkv * G, 128
    part = torch.randn(B, (Hq + 2 * Hkv) * D, device=cuda).to(dtype).float()
    cs = torch.ones(4, D // 2, 2, device=cuda)                     # pre-rotated: not read
    k1, v1 = kc.clone(), vc.clone()
    for b, n in enumerate(L):
        at = (bt[b, (n - 1) // bs].long(), slice(None), (n - 1) % bs)
        k1[at], v1[at] = (part[b, Hq * D:].to(dtype).view(2, Hkv, D)[i] for i in (0, 1))
    q = part[:, :Hq * D].to(dtype).view(B, 1, Hq, D)
    refs, mags = _reference(L, k1, v1, bt, q, D ** -0.5, 0.0, window, None)
    u = torch.finfo(dtype).eps / 2
    for _ in range(2):                                             # (tickets and sums are left as they were)
        p, k2, v2 = part.clone(), kc.clone(), vc.clone()
        got = ops.attn_decode_rope(p, None, cs, (sl - 1).long(), k2, v2, bt, sl, ns, D ** -0.5, 0.0, window, Hq, D, False, 1.0,
                                   dtype, prerot=True).view(B, 1, Hq, D)
        assert torch.equal(k1, k2) and torch.equal(v1, v2) and int((p != 0).sum()) == 0
        for b in range(B):
            assert ((got[b].double() - refs[b]).abs() <= 2.1 * u * mags[b] + 1e-30).all(), (b, L[b])
    ops.check_kernel_errors(cuda)


@pytest.mark.parametrize("L,Hkv", [([70, 131, 1, 64], 32), ([896, 70, 300, 512], 32), ([70, 131, 200, 33, 512], 32),
                                   ([70, 512] * 4, 32), ([70, 512] * 4, 40), ([960, 70] * 4, 8)])
def test_few_keys_of_up_to_8_sequences_keep_one_kernel(cuda, L, Hkv):
    """q rotated ahead of the attention and in it: p is rounded beside the same maximum"""
    kc, vc, bt, sl, ns = _setup(cuda, L, max(L), Hkv, 64, torch.bfloat16)
    B, D = len(L), 128
    assert torch.ops.ipex_llm_amd.attn_decode_plan(B, Hkv, ns) == [0, 0]
    part = torch.randn(B, 3 * Hkv * D, device=cuda)
    bias = torch.randn(3 * Hkv * D, device=cuda).bfloat16()
    cs = torch.randn(max(L), D // 2, 2, device=cuda)
    q, k1, v1 = torch.empty(B, Hkv, D, dtype=torch.bfloat16, device=cuda), kc.clone(), vc.clone()
    ops.rope_kv_fused(part[None].clone(), bias, q, k1, v1, (sl - 1).long(), bt, 1, cs, Hkv, Hkv, D)
    want = ops.attn_decode(q.view(B, 1, Hkv, D), k1, v1, bt, sl, ns, D ** -0.5)
    got = ops.attn_decode_rope(part, bias, cs, (sl - 1).long(), kc, vc, bt, sl, ns, D ** -0.5, 0.0, 0, Hkv, D, False, 1.0,
                               torch.bfloat16)
    assert torch.equal(k1, kc) and torch.equal(v1, vc)
    # the same sums but for the merge's order: far below the 2 ** -9 that p rounded beside another maximum is off
    assert ((got.float() - want.float().view_as(got)).norm() / want.float().norm()).item() < 1e-3
    ops.check_kernel_errors(cuda)


def test_bad_block_and_length_are_reported(cuda):
    kc, vc, bt, sl, ns = _setup(cuda, [100] * 17, 128, 8, 64, torch.bfloat16)
    q = torch.randn(17, 1, 32, 128, device=cuda).bfloat16()
    good = ops.attn_decode(q, kc, vc, bt, sl, ns, 0.1)
    ops.check_kernel_errors(cuda)
    bt2 = bt.clone()
    bt2[3, 1] = kc.shape[0] + 7                                    # the keys of that block are left out
    got = ops.attn_decode(q, kc, vc, bt2, sl, ns, 0.1)
    with pytest.raises(RuntimeError):
        ops.check_kernel_errors(cuda)
    keep = [b for b in range(17) if b != 3]
    assert torch.equal(got.view(17, -1)[keep], good.view(17, -1)[keep]) and got.isfinite().all()
    sl2 = sl.clone()
    sl2[5] = 1000                                                  # beyond its blocks: cut off
    ops.attn_decode(q, kc, vc, bt, sl2, ns, 0.1)
    with pytest.raises(RuntimeError):
        ops.check_kernel_errors(cuda)
