"""A decode step's state from tokens and positions in one launch: the values that separate torch ops give."""
import pytest
import torch

import ipex_llm_amd.ops as ops

pytestmark = pytest.mark.gpu


def _call(ids, pos, off, bt, bs):
    out = [torch.full_like(pos, -7) for _ in range(4)]
    lens = torch.full(pos.shape, -7, dtype=torch.int32, device=pos.device)
    torch.ops.ipex_llm_amd.decode_set_state(ids, pos, off, out[0], out[1], out[2], bt, bs, out[3], lens)
    return [t.tolist() for t in (*out, lens)]


@pytest.mark.parametrize("B", [1, 63, 64, 65, 200])
@pytest.mark.parametrize("with_off", [False, True])
def test_state(B, with_off):
    ops.require()
    dev, bs, nb = torch.device("cuda"), 16, 9
    g = torch.Generator().manual_seed(B)
    ids = torch.randint(0, 1 << 40, (B,), generator=g)
    ci = torch.randint(0, bs * nb, (B,), generator=g)
    ci[0], ci[-1] = 0, bs * nb - 1                     # first and last position of a row
    off = torch.randint(0, 5000, (B,), generator=g) if with_off else torch.zeros(B, dtype=torch.long)
    bt = torch.randint(0, 10000, (B, nb), generator=g, dtype=torch.int32)
    ops.check_kernel_errors(dev)
    got = _call(ids.to(dev), (ci + off).to(dev), off.to(dev) if with_off else None, bt.to(dev), bs)
    slots = torch.gather(bt, 1, (ci // bs)[:, None]).squeeze(1).long() * bs + ci % bs
    assert got == [ids.tolist(), (ci + off).tolist(), off.tolist(), slots.tolist(), (ci + 1).tolist()]
    assert ops.check_kernel_errors(dev) == 0


def test_outside_the_block_table():
    ops.require()
    dev = torch.device("cuda")
    ops.check_kernel_errors(dev)
    pos = torch.tensor([31, 32, 3], device=dev)
    off = torch.tensor([0, 0, 4], device=dev)
    bt = torch.tensor([[3, 4], [5, 6], [7, 8]], dtype=torch.int32, device=dev)
    got = _call(torch.zeros(3, dtype=torch.long, device=dev), pos, off, bt, 16)
    assert got[3] == [4 * 16 + 15, -1, -1] and got[4] == [32, 33, 0]
    with pytest.raises(ops.KernelError, match="sequence length"):
        ops.check_kernel_errors(dev)


def test_wrong_lengths_are_refused():
    ops.require()
    dev = torch.device("cuda")
    two, three = torch.zeros(2, dtype=torch.long, device=dev), torch.zeros(3, dtype=torch.long, device=dev)
    bt = torch.zeros(2, 4, dtype=torch.int32, device=dev)
    lens = torch.zeros(2, dtype=torch.int32, device=dev)
    with pytest.raises(RuntimeError):
        torch.ops.ipex_llm_amd.decode_set_state(three, two, None, two.clone(), two.clone(), two.clone(), bt, 16,
                                                two.clone(), lens)


def test_step_takes_every_form_of_state():
    """int32 or host tensors, scalars, the step's own tensors: the separate copies; int64 of the GPU: the launch"""
    from transformers import LlamaConfig
    from ipex_llm_amd.engine.runner import Engine
    from ipex_llm_amd.models.builder import random_native_model
    dev = torch.device("cuda")
    cfg = LlamaConfig(vocab_size=512, hidden_size=256, intermediate_size=512, num_hidden_layers=1, num_attention_heads=2,
                      num_key_value_heads=1, max_position_embeddings=512)
    eng = Engine(random_native_model(cfg, "sym_int4", dev, torch.bfloat16, seed=0))
    eng._ensure_cache(2, 128)
    st = eng.decode_step_obj([eng.new_sequence(128) for _ in range(2)], 128, True, False)
    ids, pos = torch.tensor([5, 9], device=dev), torch.tensor([70, 3], device=dev)

    def state():
        return [t.tolist() for t in (st.ids, st.pos, st.off, st.slots, st.seq_lens)]
    st.set_state(ids, pos)
    want = state()
    st.off.fill_(3)
    for i, p in ((ids.int(), pos.int()), (ids.cpu(), pos.cpu()), (torch.stack([ids, ids], 1)[:, 0], pos)):
        st.set_state(i, p)
        assert state() == want
    st.set_state(st.ids, st.pos)
    assert state() == want
    st.set_state(torch.tensor(5, device=dev), pos)
    assert state()[0] == [5, 5]
    st.set_state(ids, pos, torch.tensor([64, 0], device=dev))
    assert state()[2] == [64, 0] and state()[4] == [7, 4]
    with pytest.raises(RuntimeError):
        st.set_state(torch.zeros(3, dtype=torch.long, device=dev), pos)
