"""A prompt's down / o projection that leaves its slabs to the norm: not where the program watches the module's calls."""
from types import SimpleNamespace

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

import ipex_llm_amd.ops as ops
from ipex_llm_amd.models.decoder import NativeCausalLM
from ipex_llm_amd.transformers.low_bit_linear import LowBitLinear


@pytest.mark.parametrize("how", ["none", "hook", "pre_hook", "all_modules", "own_forward"])
def test_watched_projections_are_called(how):
    ops.require()
    seen = []
    me = SimpleNamespace(spec=SimpleNamespace(rms_eps=1e-5, norm_unit_offset=False), tp_group=None, _tp_ok=lambda p: True)
    with FakeTensorMode():
        proj = LowBitLinear(4096, 2048, "sym_int4", bias=False, device="cuda")
        x, res = (torch.empty(128, n, dtype=torch.bfloat16, device="cuda") for n in (4096, 2048))
        w, handle = torch.empty(2048, dtype=torch.bfloat16, device="cuda"), None
        if how == "hook":
            handle = proj.register_forward_hook(lambda *a: seen.append(1))
        elif how == "pre_hook":
            handle = proj.register_forward_pre_hook(lambda *a: seen.append(1))
        elif how == "all_modules":
            handle = torch.nn.modules.module.register_module_forward_hook(lambda m, *a: seen.append(m))
        elif how == "own_forward":
            call = proj.forward
            proj.forward = lambda t: (seen.append(1), call(t))[1]
        try:
            y = NativeCausalLM._proj_residual_norm(me, x, proj, res, w)
        finally:
            if handle is not None:
                handle.remove()
    assert y.shape == (128, 2048) and len(seen) == (how != "none")
