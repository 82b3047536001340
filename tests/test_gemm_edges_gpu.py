"""Products whose K is no multiple of the LDS ring's 32-k step, or whose
m/n-contiguous rows end inside a 16-byte chunk: the ring's masked last step,
repacked operands, padded rows of split partials and unaligned output rows.
Operands are small integers (every sum exact in float32 and in the result), and
what lies past their rows is NaN, so a chunk read past K shows."""
from __future__ import annotations

import pytest
import torch

from tests.kernel_names import kernels
from torchvulkan_amd import _abi

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


def operand(rows, cols, dtype, seed, pad):
    """A [rows, cols] view of rows `pad` elements wider, the rest NaN; about 1 value in 8 nonzero."""
    g = torch.Generator().manual_seed(seed)
    v = torch.randint(-1, 2, (rows, cols), generator=g) * (torch.randint(0, 8, (rows, cols), generator=g) == 0)
    wide = torch.full((rows, cols + pad), float("nan"), dtype=dtype)
    wide[:, :cols] = v.to(dtype)
    return wide.to(DEV)[:, :cols]


def product(layout, m, n, k, dtype, pad=0, bias=False, act=_abi.TVK_ACT_NONE, out_pad=0):
    # (rows padded by 8 stay 16-byte aligned where the extent is)
    a = operand(k, m, dtype, 1, pad).t() if layout == "tn" else operand(m, k, dtype, 1, pad)
    b = operand(n, k, dtype, 2, pad).t() if layout == "nt" else operand(k, n, dtype, 2, pad)
    want = (a.double() @ b.double()).cpu()
    kw = {}
    if bias:
        bv = torch.arange(n).remainder(7).sub(3).to(dtype)
        kw = {"bias": bv.to(DEV), "alpha": 2.0, "beta": 1.0, "activation": act}
        want = 2 * want + bv.double()
        if act == _abi.TVK_ACT_RELU:
            want = want.clamp(min=0)
    assert want.abs().max() <= 256
    c = torch.full((m, n + out_pad), 9, dtype=dtype, device=DEV)
    _abi.gemm(a, b, c[:, :n], **kw)
    torch.cuda.synchronize()
    assert torch.equal(c[:, :n].cpu().double(), want), _abi.gemm_plan(a, b, c[:, :n], **kw)
    assert (c[:, n:] == 9).all()
    return _abi.gemm_plan(a, b, c[:, :n], **kw)


# K past a multiple of 32 by 8, 16, 24 (masked), by an odd number (repacked), and below one step; more tiles of
# 128x128 than the 64x64 rule takes
@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
@pytest.mark.parametrize("k", [40, 1032, 1048, 1077, 1304])
def test_k_edges(gpu, layout, k):
    dtype = torch.float16 if k % 16 else torch.bfloat16
    product(layout, 1500, 1544, k, dtype)
    product(layout, 1500, 1544, k, dtype, pad=8)


@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
@pytest.mark.parametrize("m,n,k", [(1501, 1537, 1024), (1537, 1499, 1000), (1300, 2001, 93)])
def test_row_edges(gpu, layout, m, n, k):
    # (GELU's values are not exact: covered by the GEMM tests)
    for bias, act in ((False, _abi.TVK_ACT_NONE), (True, _abi.TVK_ACT_RELU)):
        product(layout, m, n, k, torch.float16, bias=bias, act=act)
    product(layout, m, n, k, torch.bfloat16, out_pad=3)


# a row's last chunk of 1 to 7 elements, in each of the ring's epilogues (none, ReLU and a bias, a bias off 16-byte
# rows), between guard columns
@pytest.mark.parametrize("n", range(1545, 1552))
def test_row_tails(gpu, n):
    plan = product("nn", 1500, n, 1032, torch.float16, out_pad=1)
    product("tn", 1504, n, 72, torch.bfloat16, out_pad=2)
    product("nn", 1500, n, 1032, torch.bfloat16, bias=True, out_pad=5)
    product("nn", 1500, n, 1024, torch.float16, bias=True, act=_abi.TVK_ACT_RELU, out_pad=3)
    assert plan == "gemm16_mfma_128x128"


# split K with a masked end in the last chunk; N no multiple of 4 (padded rows of partials)
@pytest.mark.parametrize("layout", ["nn", "tn", "nt"])
@pytest.mark.parametrize("n", [640, 637])
@pytest.mark.parametrize("k", [2056, 4088, 3001])
def test_split_edges(gpu, layout, n, k):
    plan = product(layout, 500, n, k, torch.float16)
    assert plan.endswith("_splitk")
    product(layout, 500, n, k, torch.bfloat16, bias=True, act=_abi.TVK_ACT_RELU)


# 256x256 and 128x256 tiles (whole and half rounds)
@pytest.mark.parametrize("layout", ["nn", "nt", "tn"])
@pytest.mark.parametrize("m,n,k", [(4096, 3001, 72), (3848, 3592, 200), (6000, 4500, 104)])
def test_large_tiles(gpu, layout, m, n, k):
    product(layout, m, n, k, torch.float16)
    product(layout, m, n, k, torch.bfloat16, bias=True)


def test_batches(gpu):
    # a batch whose matrices end on masked chunks and straddling columns, one and two batch dimensions
    dtype = torch.float16
    g = torch.Generator().manual_seed(4)
    a = torch.randint(-1, 2, (6, 700, 104), generator=g).to(dtype)
    b = torch.randint(-1, 2, (6, 104, 1003), generator=g).to(dtype)
    want = a.double() @ b.double()
    c = torch.empty((6, 700, 1003), dtype=dtype, device=DEV)
    _abi.gemm(a.to(DEV), b.to(DEV), c)
    c4 = torch.empty((2, 3, 700, 1003), dtype=dtype, device=DEV)
    _abi.gemm(a.to(DEV).view(2, 3, 700, 104), b.to(DEV).view(2, 3, 104, 1003), c4)
    torch.cuda.synchronize()
    assert torch.equal(c.cpu().double(), want) and torch.equal(c4.cpu().double().view(6, 700, 1003), want)


# which kernel runs under the plan's name: the ring (and its tile) or the register-staged kernel, on both sides of the
# lines. m, n, k, batch, layout, ring tile
@pytest.mark.parametrize("m,n,k,batch,layout,tile", [
    (1500, 1544, 1040, 1, "nn", "128, 128"), (1500, 1544, 40, 1, "nn", "128, 128"), (1500, 1544, 24, 1, "nn", None),
    (1501, 1537, 1024, 1, "nn", "128, 128"), (1501, 1537, 1024, 1, "tn", "128, 128"),
    (1500, 1544, 1016, 1, "nt", None), (1500, 1544, 1032, 1, "nt", "128, 128"),   # two k-contiguous operands: from 1024
    (2048, 2048, 1032, 1, "nt", "128, 128"), (2049, 2048, 1032, 1, "nt", None),   # to 256 tiles
    (1280, 2064, 1032, 3, "nt", None), (3000, 3000, 1032, 1, "nt", "256, 256"), (4352, 104, 1032, 16, "nt", None),
    (500, 640, 2056, 1, "nn", "128, 128"), (500, 640, 2056, 1, "nt", None),       # split K
    (4096, 3008, 72, 1, "nt", "256, 256"), (4600, 4600, 104, 1, "nn", "128, 256"),
])
def test_kernel_of_a_plan(gpu, m, n, k, batch, layout, tile):
    dtype = torch.float16
    sh = (batch,) if batch > 1 else ()
    a = torch.ones((*sh, k, m), dtype=dtype, device=DEV).transpose(-1, -2) if layout == "tn" else torch.ones((*sh, m, k), dtype=dtype, device=DEV)
    b = torch.ones((*sh, n, k), dtype=dtype, device=DEV).transpose(-1, -2) if layout == "nt" else torch.ones((*sh, k, n), dtype=dtype, device=DEV)
    c = torch.empty((*sh, m, n), dtype=dtype, device=DEV)
    assert _abi.gemm_plan(a, b, c).startswith("gemm16_mfma_")
    names = [x for x in kernels(lambda: _abi.gemm(a, b, c)) if "gemm16_" in x]
    assert len(names) == 1 and ("gemm16_dma_kernel" in names[0]) == (tile is not None), names
    assert tile is None or f", {tile}, 4, " in names[0], names
    assert (c == k).all()
