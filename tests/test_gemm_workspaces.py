"""Where products that are cut over k leave their partial sums: never where another stream, thread or captured graph does."""
import gc
import threading
import weakref
from types import SimpleNamespace

import pytest
import torch

from infer_amd import ops

MIB = 1 << 20


class Streams:
    """Stands in for the streams of a GPU; memory comes from the host."""
    def __init__(self, monkeypatch):
        self.handle, self.capturing = 1, 0
        empty = torch.empty
        monkeypatch.setattr(ops, "_gemm_workspaces", type(ops._gemm_workspaces)())
        monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: self.capturing != 0)
        monkeypatch.setattr(ops._lib, "load", lambda: SimpleNamespace(infer_stream_capture_id=lambda stream: self.capturing))
        monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
        monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: SimpleNamespace(cuda_stream=self.handle))
        monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda index: self.handle, raising=False)
        monkeypatch.setattr(torch, "empty", lambda *size, device=None, **kw: empty(*size, **kw))

    def workspace(self, handle, need=MIB, capturing=0, device="cuda:0"):
        self.handle, self.capturing = handle, capturing
        return ops._gemm_workspace(device, need)


@pytest.fixture
def streams(monkeypatch):
    return Streams(monkeypatch)


def apart(*workspaces):
    return len({w.data_ptr() for w in workspaces}) == len(workspaces)


def test_a_stream_keeps_its_workspace(streams):
    a, b = streams.workspace(11), streams.workspace(12)
    assert apart(a, b)
    assert streams.workspace(11) is a and streams.workspace(12) is b
    assert streams.workspace(11, device="cuda") is a                   # the current device by another name
    assert streams.workspace(11, 2 * a.numel()).numel() >= 2 * a.numel()
    assert streams.workspace(11, 0) is None


def test_captured_products_share_with_nobody(streams):
    """Two streams of one capture run side by side, and so do two graphs that are replayed on different streams, or a graph and eager work."""
    eager = streams.workspace(21)
    captured = [streams.workspace(22, capturing=1), streams.workspace(23, capturing=1), streams.workspace(22, capturing=2)]
    assert apart(eager, *captured)
    assert streams.workspace(22, capturing=2) is captured[2] and streams.workspace(21) is eager
    assert apart(eager, streams.workspace(21, capturing=3))


def test_threads_on_one_stream_share_with_nobody(streams):
    """A product and the sum of its pieces are two launches, and another thread's product may come between them."""
    mine, theirs = streams.workspace(31), []
    t = threading.Thread(target=lambda: theirs.append(streams.workspace(31)))
    t.start()
    t.join()
    assert apart(mine, *theirs)


def test_memory_of_streams_out_of_use_is_given_back(streams):
    first = weakref.ref(streams.workspace(41))
    kept = [streams.workspace(42 + i) for i in range(8)]
    gc.collect()
    assert first() is None
    kept = [weakref.ref(w) for w in kept]
    gc.collect()
    assert 1 <= sum(w() is not None for w in kept) <= 4
    seen = []
    t = threading.Thread(target=lambda: seen.append(weakref.ref(streams.workspace(41))))
    t.start()
    t.join()
    gc.collect()
    assert seen[0]() is None


# ------------------------------------------------------------------ on the GPU
def operands(gpu, seed):
    """Small integers, whose sums are exact, so that any mix of two products shows; cut over k (1024 rows of weights)."""
    g = torch.Generator(device=gpu).manual_seed(seed)
    x = torch.randint(-1, 2, (8, 4096), generator=g, device=gpu).to(torch.bfloat16)
    w = (torch.randint(-1, 2, (1024, 4096), generator=g, device=gpu) * (torch.rand((1024, 4096), generator=g, device=gpu) < 0.5)).to(torch.bfloat16)
    assert ops._lib.load().infer_skinny_gemm_workspace_bytes(8, 1024, 4096) > 0
    return x, w, x.float() @ w.float().t()


@pytest.mark.gpu
def test_forked_streams_of_a_capture(gpu):
    (x, w, want), (y, v, wanted) = operands(gpu, 1), operands(gpu, 2)
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    ops.linear(x, w)
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        here = torch.cuda.current_stream()
        side.wait_stream(here)
        a = [ops.linear(x, w) for _ in range(8)]
        with torch.cuda.stream(side):
            b = [ops.linear(y, v) for _ in range(8)]
        here.wait_stream(side)
    for _ in range(5):
        for t in a + b:
            t.zero_()
        assert torch.equal(ops.linear(-x, w).float(), -want)            # eager work between the replays
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(t.float(), want) for t in a) and all(torch.equal(t.float(), wanted) for t in b)


@pytest.mark.gpu
def test_graphs_replayed_on_two_streams(gpu):
    sets = [operands(gpu, 3), operands(gpu, 4)]
    streams, graphs, outs = [torch.cuda.Stream() for _ in sets], [torch.cuda.CUDAGraph() for _ in sets], []
    ops.linear(*sets[0][:2])
    torch.cuda.synchronize()
    for graph, (x, w, _) in zip(graphs, sets):
        with torch.cuda.graph(graph):
            outs.append([ops.linear(x, w) for _ in range(8)])
    for _ in range(5):
        for t in outs[0] + outs[1]:
            t.zero_()
        torch.cuda.synchronize()
        for graph, stream in zip(graphs, streams):
            with torch.cuda.stream(stream):
                graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(t.float(), want) for out, (_, _, want) in zip(outs, sets) for t in out)
