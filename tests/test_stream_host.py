"""The current stream's handle comes from torch's public interface where the faster private call is missing."""

import types

import torch

from gaudi_kernels import ops


def test_stream_without_the_private_call(monkeypatch):
    monkeypatch.setattr(ops, "_raw_stream", None)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device: types.SimpleNamespace(cuda_stream=7 + device.index))
    assert ops._stream(torch.device("cuda", 2)) == 9


def test_stream_private_call(monkeypatch):
    monkeypatch.setattr(ops, "_raw_stream", lambda index: 100 + index)
    assert ops._stream(torch.device("cuda", 1)) == 101
