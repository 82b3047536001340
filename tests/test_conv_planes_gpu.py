"""Channels-last convolution paths on planes that are no whole number of
32-pixel stages or 8-pixel runs: the layout copy's unaligned and partial runs,
and the grad weight over channels-last dy. Operands are small integers, so that
every sum is exact in float32 and in the 16-bit results whatever its order: a
dropped, repeated or misplaced pixel, tap or channel changes a value."""
from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

from torchvulkan_amd import _abi

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


def ints(shape, seed, lo, hi):
    return torch.randint(lo, hi + 1, shape, generator=torch.Generator().manual_seed(seed)).double()


# batch, cin, cout, (h, w), kernel, stride, dilation: pixels below, at and above one stage and one 8-pixel run;
# column tiles of 64, 128 and 256 with a remainder; rows (taps x channels) past one 256-row tile; 1x1; a plane per pixel
CASES = [
    (3, 32, 64, (7, 7), 3, 1, 1),
    (2, 64, 128, (14, 14), 3, 1, 1),
    (2, 32, 264, (28, 28), 3, 1, 1),
    (5, 96, 72, (9, 5), 3, 2, 1),
    (2, 32, 40, (27, 27), 3, 2, 1),
    (1, 64, 64, (33, 31), 3, 1, 2),
    (7, 32, 136, (14, 14), 1, 1, 1),
    (6, 32, 32, (7, 7), 1, 2, 1),
    (40, 32, 32, (1, 1), 1, 1, 1),
    (2, 8, 16, (6, 11), 3, 1, 1),
]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_every_direction(gpu, dtype, case):
    n, cin, cout, (h, w), k, stride, dil = CASES[case]
    pad = dil * (k // 2)
    x = ints((n, cin, h, w), case, -1, 1)
    wt = ints((cout, cin, k, k), case + 50, -1, 1) * (ints((cout, cin, k, k), case + 60, 0, 3) == 0)
    y = F.conv2d(x, wt, stride=stride, padding=pad, dilation=dil)
    dy = ints(y.shape, case + 70, -1, 1) * (ints(y.shape, case + 80, 0, 3) == 0)
    dx = torch.nn.grad.conv2d_input(x.shape, wt, dy, stride=stride, padding=pad, dilation=dil)
    dw = torch.nn.grad.conv2d_weight(x, wt.shape, dy, stride=stride, padding=pad, dilation=dil)
    top = 256 if dtype == torch.bfloat16 else 2048
    assert max(t.abs().max().item() for t in (y, dx, dw)) <= top   # exact in the dtype
    xd, wd, dyd = (t.to(dtype).to(DEV) for t in (x, wt, dy))
    got = (_abi.conv2d_fwd(xd, wd, stride=stride, padding=pad, dilation=dil),
           _abi.conv2d_dgrad(dyd, wd, tuple(x.shape), stride=stride, padding=pad, dilation=dil),
           _abi.conv2d_wgrad(xd, dyd, tuple(wt.shape), stride=stride, padding=pad, dilation=dil))
    torch.cuda.synchronize()
    for g, want, name in zip(got, (y, dx, dw), ("y", "dx", "dw")):
        assert torch.equal(g.cpu().double(), want), f"{name} of case {CASES[case]} {dtype}"


def test_every_family_of_an_odd_plane(gpu):
    # the channels-last grad weight is offered where whole 8-channel chunks allow it, and each family agrees
    x, dy = (ints(s, i, -1, 1).half().to(DEV) for i, s in enumerate([(2, 32, 14, 14), (2, 24, 14, 14)]))
    dw = torch.empty((24, 32, 3, 3), dtype=torch.float16, device=DEV)
    d = _abi.conv_problem(x, dw, dy, padding=1)
    names = _abi.conv_candidates(d, _abi.TVK_CONV_WGRAD)
    assert names == ["conv_ring", "conv_implicit_gemm"]
    want = torch.nn.grad.conv2d_weight(x.cpu().double(), dw.shape, dy.cpu().double(), padding=1)
    for name in names:
        _abi.conv_choose(d, _abi.TVK_CONV_WGRAD, name)
        dw.fill_(7)
        _abi.conv_run(d, _abi.TVK_CONV_WGRAD)
        torch.cuda.synchronize()
        assert torch.equal(dw.cpu().double(), want), name
    _abi.tune_reset()


def test_captured_grad_weight(gpu):
    # a captured call allocates nothing: on a stream whose workspace pool is empty, a short reduction is captured,
    # replayed between eager calls, and gives the eager result every time
    x, dy = (ints(s, i, -1, 1).half().to(DEV) for i, s in enumerate([(2, 32, 14, 14), (2, 24, 14, 14)]))
    want = torch.nn.grad.conv2d_weight(x.cpu().double(), (24, 32, 3, 3), dy.cpu().double(), padding=1)
    dw = torch.empty((24, 32, 3, 3), dtype=torch.float16, device=DEV)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
        d = _abi.conv_problem(x, dw, dy, padding=1)
        _abi.conv_run(d, _abi.TVK_CONV_WGRAD)
    for _ in range(3):
        dw.zero_()
        graph.replay()
        eager = _abi.conv2d_wgrad(x, dy, (24, 32, 3, 3), padding=1)
        torch.cuda.synchronize()
        assert torch.equal(dw.cpu().double(), want) and torch.equal(eager.cpu().double(), want)
