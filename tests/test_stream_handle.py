"""The stream handle of the binding: torch's private accessor where there is one, the public one else."""

import types

import torch

import w4a16


def test_private_accessor_and_fallback(monkeypatch):
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 3)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: types.SimpleNamespace(cuda_stream=77))
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda device: 40 + device, raising=False)
    assert w4a16._stream(None) == 43
    monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream")
    assert w4a16._stream(None) == 77
    assert w4a16._stream(5) == 5
    assert w4a16._stream(types.SimpleNamespace(cuda_stream=6)) == 6
