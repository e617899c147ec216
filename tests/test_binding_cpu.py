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
