"""Captured calls that need scratch (split-K partials, repacked operands, the
streaming kernels', convolution and reduction partials, the attention delta):
the memory belongs to the graph. Replays on other streams stay right while
eager calls on the capture's stream use, grow and trim the pool, and the memory
is given back after the graph. (The pool's rules are checked on the CPU,
test_scratch_pool.py.)"""
from __future__ import annotations

import ctypes as C
import gc
import time

import pytest
import torch

from torchvulkan_amd import _abi

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


def rand(*shape, seed=0, dtype=torch.float16):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)).to(dtype).to(DEV)


def gemm_call(m, n, k, nt):
    a, b = rand(m, k, seed=m), rand(n, k, seed=n).t() if nt else rand(k, n, seed=n)
    return lambda out: _abi.gemm(a, b, out), torch.empty((m, n), dtype=torch.float16, device=DEV)


def wgrad_call():
    x, dy = rand(8, 64, 32, 32, seed=1), rand(8, 64, 32, 32, seed=2)
    dw = torch.empty((64, 64, 3, 3), dtype=torch.float16, device=DEV)

    def run(out):
        _abi.conv_run(_abi.conv_problem(x, out, dy, padding=1), _abi.TVK_CONV_WGRAD)

    return run, dw


CALLS = {
    "split tiles": lambda: gemm_call(256, 512, 8192, False),
    "repacked operands": lambda: gemm_call(999, 777, 1001, False),
    "few rows, k-contiguous": lambda: gemm_call(33, 256, 8000, True),
    "few rows, n-contiguous": lambda: gemm_call(16, 1024, 8192, False),
    "conv grad weight": wgrad_call,
}


def reserved() -> int:
    v = C.c_size_t(0)
    _abi.check(_abi.load().tvk_memory_reserved(0, C.byref(v)))
    return v.value


def trim():
    _abi.check(_abi.load().tvk_empty_cache(0))


def test_replays_beside_eager_calls(gpu):
    # one graph of all calls, captured on a stream whose pool is cold, replayed on a second stream while the first
    # runs the same calls eagerly, grows the pool and trims it
    calls = {name: make() for name, make in CALLS.items()}
    want = {}
    for name, (run, out) in calls.items():
        want[name] = torch.empty_like(out)
        run(want[name])
    torch.cuda.synchronize()
    home, other, graph = torch.cuda.Stream(), torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=home):
        for run, out in calls.values():
            run(out)
    eager = {name: torch.empty_like(out) for name, (_, out) in calls.items()}
    large = gemm_call(2048, 2048, 4104, False)   # more scratch than any of them: the stream's pool grows
    for step in range(6):
        with torch.cuda.stream(other):
            for _, out in calls.values():
                out.fill_(7)
            for _ in range(3):
                graph.replay()
        with torch.cuda.stream(home):
            for _ in range(2):
                for name, (run, _) in calls.items():
                    run(eager[name])
            if step % 2:
                large[0](large[1])
        if step % 3 == 2:
            trim()
        torch.cuda.synchronize()
        for name, (_, out) in calls.items():
            assert torch.equal(out, want[name]), f"step {step}: {name}, replayed"
            assert torch.equal(eager[name], want[name]), f"step {step}: {name}, eager"


def test_two_graphs_of_one_stream(gpu):
    # each has its own memory: they may be replayed at the same time
    stream, graphs, outs = torch.cuda.Stream(), [], []
    calls = [gemm_call(33, 256, 8000, True), gemm_call(40, 256, 6000, True)]
    want = [torch.empty_like(o) for _, o in calls]
    for (run, _), w in zip(calls, want):
        run(w)
    torch.cuda.synchronize()
    for run, out in calls:
        graphs.append(torch.cuda.CUDAGraph())
        outs.append([torch.empty_like(out) for _ in range(10)])
        with torch.cuda.graph(graphs[-1], stream=stream):
            for o in outs[-1]:
                run(o)
    streams = [torch.cuda.Stream() for _ in graphs]
    for _ in range(4):
        for g, st in zip(graphs, streams):
            with torch.cuda.stream(st):
                g.replay()
        torch.cuda.synchronize()
        for i in range(2):
            assert all(torch.equal(o, want[i]) for o in outs[i])


def test_memory_returns_with_the_graph(gpu):
    torch.cuda.synchronize()
    gc.collect()
    run, out = gemm_call(256, 512, 8192, False)
    trim()
    before = reserved()
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        run(out)
    held = reserved()
    assert held > before
    trim()
    assert reserved() == held   # the graph's
    graph.replay()
    torch.cuda.synchronize()
    del graph
    gc.collect()
    # the runtime tells when the last launch is behind it, which it may notice with the next one
    for _ in range(200):
        out.zero_()
        torch.cuda.synchronize()
        trim()
        if reserved() < held:
            break
        time.sleep(0.01)
    assert reserved() <= before
