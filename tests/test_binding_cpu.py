"""The Python binding's host side, without a device."""
from types import SimpleNamespace

import pytest
import torch

import helpers


@pytest.fixture()
def binding():
    return helpers.load_sgq()


def test_stream_handle_without_the_raw_query(binding, monkeypatch):
    """A torch that lacks the non-public raw-stream query gives the handle of its
    public current stream."""
    monkeypatch.setattr(binding, "_raw_stream", None)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device: SimpleNamespace(cuda_stream=1000 + device.index))
    assert binding._stream(torch.device("cuda:3")) == 1003


def test_stream_handle_of_the_current_device(binding, monkeypatch):
    monkeypatch.setattr(binding, "_raw_stream", lambda index: 2000 + index)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 5)
    assert binding._stream(torch.device("cuda:3")) == 2003
    assert binding._stream(torch.device("cuda")) == 2005


class Tagged(torch.Tensor):
    pass


@pytest.mark.parametrize("kind", [torch.Tensor, Tagged, torch.nn.Parameter])
def test_outputs_are_plain_tensors(binding, kind):
    x = torch.zeros(3, 4)
    x = x.as_subclass(kind) if kind is Tagged else (torch.nn.Parameter(x) if kind is torch.nn.Parameter else x)
    y = binding._new_output(x, 3, 7)
    assert type(y) is torch.Tensor and y.shape == (3, 7) and y.dtype == torch.float32 and not y.requires_grad
