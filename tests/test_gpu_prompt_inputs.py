"""A prompt's host tensors travel in one copy: values, types and shapes arrive as they were, beside what is on the device."""
import pytest
import torch

from ipex_llm_amd.engine.runner import _to_device

PARTS = [torch.arange(7), torch.tensor([3], dtype=torch.int32), torch.zeros(1, 0, dtype=torch.int32), torch.arange(10, dtype=torch.int32).view(2, 5),
         torch.arange(12).view(3, 4).t(), torch.tensor([1.5, -2.0], dtype=torch.float16)]


def _check(dev):
    there = torch.arange(5, device=dev)
    *got, same = _to_device(dev, PARTS + [there])
    assert same.data_ptr() == there.data_ptr()
    for g, p in zip(got, PARTS):
        assert g.device.type == torch.device(dev).type and g.dtype == p.dtype and g.shape == p.shape and torch.equal(g.cpu(), p)


def test_host():
    _check("cpu")


@pytest.mark.gpu
def test_device(cuda):
    _check(cuda)
    assert all(g.is_contiguous() for g in _to_device(cuda, PARTS))
