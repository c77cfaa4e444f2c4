"""The handle that calls without a stream argument launch on is the current stream's."""
from __future__ import annotations

import types

import pytest


def test_handle_without_the_private_accessor(monkeypatch):
    """torch's accessor of the raw handle is private: a torch without it serves through current_stream."""
    import torch

    from qwowl35_amd import runtime as rt

    monkeypatch.setattr(torch.cuda, "current_stream", lambda device: types.SimpleNamespace(cuda_stream=4096 + device))
    assert rt._raw_stream_of(types.SimpleNamespace())(2) == 4098
    monkeypatch.setattr(rt, "_raw_stream", rt._raw_stream_of(types.SimpleNamespace()))
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 3)
    assert rt._stream(None).value == 4099
    assert rt._stream(types.SimpleNamespace(cuda_stream=7)).value == 7


@pytest.mark.gpu
def test_handle_follows_the_current_stream(cuda):
    import torch

    from qwowl35_amd import runtime as rt

    side = torch.cuda.Stream()
    assert (rt._stream(None).value or 0) == torch.cuda.current_stream().cuda_stream
    with torch.cuda.stream(side):
        assert rt._stream(None).value == side.cuda_stream
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        assert rt._stream(None).value == torch.cuda.current_stream().cuda_stream
