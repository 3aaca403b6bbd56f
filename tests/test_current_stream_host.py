"""The current stream's handle where torch does not export its raw form.  No GPU."""
import types

import torch

from holoflow_amd import hfx


def test_a_torch_without_the_raw_handle(monkeypatch):
    monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream", raising=False)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch.cuda, "Stream", types.SimpleNamespace)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: types.SimpleNamespace(cuda_stream=4096))
    assert hfx._stream(None).value == 4096


def test_the_raw_handle_where_there_is_one(monkeypatch):
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 3)
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda device: 1000 + device, raising=False)
    assert hfx._stream(None).value == 1003
