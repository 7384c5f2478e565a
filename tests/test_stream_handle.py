"""The stream that a call without one is given: torch's current stream, also by a torch build that lacks the
undocumented call for its handle.  CPU only (the device queries are replaced)."""
from __future__ import annotations

import types

import pytest
import torch

from voxelrt_amd import api


@pytest.mark.parametrize("raw", [None, lambda device: 1000 + device])
def test_current_stream(monkeypatch, raw):
    monkeypatch.setattr(torch.cuda, "is_available", lambda: True)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 3)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: types.SimpleNamespace(cuda_stream=1003))
    monkeypatch.setattr(api, "_raw_stream", raw)
    assert api._stream_handle(None) == 1003


def test_without_a_device_and_given(monkeypatch):
    monkeypatch.setattr(torch.cuda, "is_available", lambda: False)
    assert api._stream_handle(None) == 0
    assert api._stream_handle(77) == 77


@pytest.mark.gpu
def test_handles_agree(cuda):
    for stream in (torch.cuda.current_stream(), torch.cuda.Stream()):
        with torch.cuda.stream(stream):
            assert api._stream_handle(None) == stream.cuda_stream == api._stream_handle(stream)
