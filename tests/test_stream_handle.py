"""The stream that the Python entry points launch on: the current one, by the handle that torch gives directly or, where
it does not (or nothing has touched the GPU yet), through the Stream object; an explicit stream as an object or a
handle."""
from types import SimpleNamespace

import pytest
import torch

from conftest import announce
from g4attn import ops


def test_current_stream_paths(monkeypatch):
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: SimpleNamespace(cuda_stream=1001))
    monkeypatch.setattr(ops, "_current_device", lambda: 3)
    monkeypatch.setattr(ops, "_raw_stream", lambda device: 70 + device)
    monkeypatch.setattr(torch.cuda, "is_initialized", lambda: True)
    assert ops._stream() == 73
    monkeypatch.setattr(torch.cuda, "is_initialized", lambda: False)
    assert ops._stream() == 1001
    monkeypatch.setattr(torch.cuda, "is_initialized", lambda: True)
    monkeypatch.setattr(ops, "_raw_stream", None)  # a torch without it
    assert ops._stream() == 1001
    assert ops._stream(SimpleNamespace(cuda_stream=5)) == 5 and ops._stream(7) == 7 and ops._stream(0) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("direct", [True, False])
def test_launches_follow_the_current_stream(dev, monkeypatch, direct):
    announce(f"argmax on the current stream, handle {'direct' if direct else 'through the object'}")
    assert ops._raw_stream is not None  # the torch in use gives the handle
    if not direct:
        monkeypatch.setattr(ops, "_raw_stream", None)
    assert ops._stream() == torch.cuda.current_stream().cuda_stream
    x = torch.arange(5000, dtype=torch.float32, device=dev)
    res = torch.full((1,), -1, dtype=torch.int32, device=dev)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        assert ops._stream() == side.cuda_stream != torch.cuda.default_stream().cuda_stream
        ops.argmax(x, res, 5000)
    side.synchronize()
    assert int(res.item()) == 4999
    res.fill_(-1)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):  # on the capturing stream, or nothing is captured
        ops.argmax(x, res, 4000)
    for _ in range(3):
        res.fill_(-1)
        graph.replay()
        torch.cuda.synchronize()
        assert int(res.item()) == 3999
