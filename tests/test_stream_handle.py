"""The raw stream handle that the Python layer hands to the library (CPU)."""
from types import SimpleNamespace

import torch

from helm3d import core


def test_raw_stream_of_the_current_device(monkeypatch):
    monkeypatch.setattr(core, "_RAW_STREAM", lambda device: 1000 + device)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 3)
    assert core._stream_ptr() == 1003


def test_public_stream_where_the_raw_call_is_missing(monkeypatch):
    monkeypatch.setattr(core, "_RAW_STREAM", None)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: SimpleNamespace(cuda_stream=77))
    assert core._stream_ptr() == 77
