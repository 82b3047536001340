"""Products of few rows with a k-contiguous weight ([N][K], nn.Linear's): the
LDS ring of gemm_skinny.hip at the edges of its stages (256 k), strips (64
columns), row blocks (16, 32, 64) and K chunks. Operands are small integers, so
every sum is exact in float32 and in the result whatever its order."""
from __future__ import annotations

import pytest
import torch

from torchvulkan_amd import _abi

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


def ints(shape, seed, lo=-1, hi=1):
    return torch.randint(lo, hi + 1, shape, generator=torch.Generator().manual_seed(seed))


def operands(m, n, k, dtype, seed, batch=()):
    x = ints((*batch, m, k), seed)
    w = ints((*batch, n, k), seed + 1) * (ints((*batch, n, k), seed + 2, 0, 7) == 0)   # sums of about sqrt(k / 12)
    return x.to(dtype), w.to(dtype)


# K: one chunk, below / at / past a stage, ragged, split with a short last chunk and a ragged end, rows 4 KB apart
# (rotated stages) unsplit and split; N: a strip, a ragged strip, no multiple of 4 (padded rows of partials)
@pytest.mark.parametrize("k", [64, 248, 256, 264, 1000, 2048, 4096, 4104, 6144])
@pytest.mark.parametrize("n", [64, 72, 130, 1000])
@pytest.mark.parametrize("m", [1, 15, 16, 17, 32, 33, 64])
def test_edges(gpu, m, n, k):
    dtype = torch.float16 if (m + n) % 2 else torch.bfloat16
    x, w = operands(m, n, k, dtype, m + n + k)
    want = x.double() @ w.double().t()
    assert want.abs().max() <= 256
    xd, wd = x.to(DEV), w.to(DEV)
    c = torch.full((m, n), 7, dtype=dtype, device=DEV)
    # (below 4 k a row, 8 from 33 rows, the tiles take more than 16 rows)
    ring = m <= 16 or k >= (4 if m <= 32 else 8) * m
    assert gpu.gemm_plan(xd, wd.t(), c).startswith("gemm16_skinny_bk" if ring else "gemm16_mfma_64x64")
    for _ in range(3):   # counters are left at zero
        _abi.gemm(xd, wd.t(), c)
    torch.cuda.synchronize()
    assert torch.equal(c.cpu().double(), want)


@pytest.mark.parametrize("m", [3, 40])
def test_views_batches_and_epilogue(gpu, m):
    # sliced rows whose next columns are NaN, two batch entries, a bias, alpha and ReLU, an output of wider rows
    dtype = torch.float16
    x, w = operands(m, 200, 520, dtype, 5, (2,))
    xd = torch.full((2, m, 536), float("nan"), dtype=dtype)
    wd = torch.full((2, 200, 528), float("nan"), dtype=dtype)
    xd[..., :520], wd[..., :520] = x, w
    xd, wd = xd.to(DEV)[..., :520], wd.to(DEV)[..., :520]
    bias = ints((200,), 9, -3, 3).to(dtype)
    out = torch.full((2, m, 208), 5, dtype=dtype, device=DEV)
    _abi.gemm(xd, wd.transpose(1, 2), out[..., :200], bias=bias.to(DEV), alpha=2.0, beta=3.0, activation=_abi.TVK_ACT_RELU)
    torch.cuda.synchronize()
    want = torch.relu(2 * (x.double() @ w.double().transpose(1, 2)) + 3 * bias.double())
    assert torch.equal(out[..., :200].cpu().double(), want)
    assert (out[..., 200:] == 5).all()


@pytest.mark.parametrize("m", [16, 64])
def test_noalloc_and_capture(gpu, m):
    # without scratch of the pool: the allocation-free entry point sums in a second launch above 16 rows, up to them,
    # and in a captured call whose stream has no idle scratch, a workgroup takes the chunks of K in turn
    dtype = torch.bfloat16
    x, w = operands(m, 512, 8192 if m == 16 else 4096, dtype, 11)
    want = x.double() @ w.double().t()
    xd, wd = x.to(DEV), w.to(DEV)
    c = torch.full((m, 512), 7, dtype=dtype, device=DEV)
    _abi.gemm_noalloc(xd, wd.t(), c)
    torch.cuda.synchronize()
    assert torch.equal(c.cpu().double(), want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        _abi.gemm(xd, wd.t(), c)
    other = torch.empty_like(c)
    for _ in range(3):
        c.fill_(7)
        graph.replay()
        _abi.gemm(xd, wd.t(), other)
        torch.cuda.synchronize()
        assert torch.equal(c.cpu().double(), want) and torch.equal(other, c)


# K chunks summed in a captured second launch: one strip and several, rows of one, two and four blocks
@pytest.mark.parametrize("m,n,k", [(17, 64, 2048), (33, 256, 8000), (64, 1000, 4096), (32, 512, 8192)])
def test_capture_on_a_warm_stream(gpu, m, n, k):
    # a stream whose pool holds an idle buffer: the captured call splits K like an eager one
    dtype = torch.bfloat16
    x, w = operands(m, n, k, dtype, 11)
    want = x.double() @ w.double().t()
    xd, wd = x.to(DEV), w.to(DEV)
    c, e = (torch.full((m, n), 7, dtype=dtype, device=DEV) for _ in range(2))
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        _abi.gemm(xd, wd.t(), e)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        _abi.gemm(xd, wd.t(), c)
    for _ in range(3):
        c.fill_(7)
        graph.replay()
        _abi.gemm(xd, wd.t(), e)
        torch.cuda.synchronize()
        assert torch.equal(c.cpu().double(), want) and torch.equal(e, c)


# real values whose sums round: the split call (K in chunks over workgroups), the allocation-free entry point and a
# captured call on a stream without idle scratch give the same bits; biases and activations in either epilogue
@pytest.mark.parametrize("m", [1, 7, 16, 17, 40, 64])
@pytest.mark.parametrize("n,k", [(64, 2048), (250, 4104), (1000, 6000), (512, 1800)])
def test_same_bits_without_partials(gpu, m, n, k):
    dtype = torch.bfloat16 if n % 4 else torch.float16
    g = torch.Generator().manual_seed(m + n)
    x, w = torch.randn((m, k), generator=g).to(dtype).to(DEV), torch.randn((n, k), generator=g).to(dtype).to(DEV)
    kw = {"bias": torch.randn((n,), generator=g).to(dtype).to(DEV), "alpha": 0.5, "beta": 2.0, "activation": _abi.TVK_ACT_GELU}
    for kw in ({}, kw):
        want, got, captured = (torch.full((m, n), 7, dtype=dtype, device=DEV) for _ in range(3))
        _abi.gemm(x, w.t(), want, **kw)
        _abi.gemm_noalloc(x, w.t(), got, **kw)
        stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=stream):
            _abi.gemm(x, w.t(), captured, **kw)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want) and torch.equal(captured, want)


# the allocation-free entry point up to 16 rows uses none of the array its calls share: calls that overlap, replayed
# from two graphs on two streams, are independent
def test_noalloc_overlapping_calls(gpu):
    m, n, k, calls = 16, 1024, 8192, 20
    x, w = operands(m, n, k, torch.bfloat16, 3)
    xs, wd = [(x * (i + 1)).to(DEV) for i in range(2)], w.to(DEV)
    outs = [torch.empty((calls, m, n), dtype=torch.bfloat16, device=DEV) for _ in range(2)]
    graphs, streams = [], [torch.cuda.Stream() for _ in range(2)]
    for j, st in enumerate(streams):
        graphs.append(torch.cuda.CUDAGraph())
        with torch.cuda.graph(graphs[j], stream=st):
            for i in range(calls):
                _abi.gemm_noalloc(xs[j], wd.t(), outs[j][i])
    want = x.double() @ w.double().t()
    for _ in range(5):
        for j, st in enumerate(streams):
            with torch.cuda.stream(st):
                outs[j].zero_()
                graphs[j].replay()
        torch.cuda.synchronize()
        for j in range(2):
            ok = (outs[j].cpu().double() == (j + 1) * want).flatten(1).all(dim=1)
            assert ok.all(), f"stream {j}: {int((~ok).sum())} of {calls} calls differ"
