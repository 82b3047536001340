"""Which products of 17 to 64 rows with a k-contiguous weight ([N][K]) the ring
of few rows takes (plan name "gemm16_skinny_bk"): both sides of each line of
its rule, from the C ABI's plan, without a GPU."""
from __future__ import annotations

import ctypes as C

import pytest

from torchvulkan_amd import _abi

RING = "gemm16_skinny_bk"


def plan(m, n, k, batch=1):
    d = _abi.GemmDesc()
    d.dtype, d.batch, d.M, d.N, d.K = _abi.TVK_F16, batch, m, n, k
    d.a = d.b = d.c = 1 << 20   # (aligned, never read)
    d.a_stride, d.b_stride, d.c_stride = _abi.I64x3(m * k, k, 1), _abi.I64x3(n * k, 1, k), _abi.I64x3(m * n, n, 1)
    d.alpha = 1.0
    name = C.create_string_buffer(128)
    assert _abi.load().tvk_gemm_plan(C.byref(d), name, 128) == _abi.TVK_OK
    return name.value.decode()


# (m, n, k, batch) the ring takes, and a neighbour across the line that it leaves to the tiles
@pytest.mark.parametrize("ring,tiles", [
    ((17, 512, 72, 1), (17, 512, 64, 1)),                # 4 k a row, 8 from 33 rows
    ((32, 512, 128, 1), (32, 512, 120, 1)),
    ((33, 512, 264, 1), (33, 512, 256, 1)),
    ((64, 512, 512, 1), (64, 512, 504, 1)),
    ((32, 16384, 1024, 1), (32, 16448, 1024, 1)),        # one round of workgroups
    ((33, 16384, 1024, 1), (33, 16448, 1024, 1)),
    ((48, 32768, 1000, 1), (48, 32832, 1000, 1)),        # two, K off the 32 grid
    ((24, 20000, 776, 1), (24, 20000, 744, 1)),
    ((24, 20000, 2040, 1), (24, 20000, 2056, 1)),
    ((32, 32000, 4096, 1), (33, 32000, 4096, 1)),        # one long wide weight
    ((24, 1024, 512, 16), (24, 1024, 512, 17)),
    ((64, 512, 1000, 32), (64, 576, 1000, 32)),
    ((20, 64, 2048, 256), (20, 64, 2048, 257)),          # batches that the tiles split too
    ((40, 64, 2048, 128), (40, 64, 2048, 129)),
    ((40, 64, 4096, 64), (40, 64, 4096, 65)),
    ((32, 512, 8184, 16), (32, 512, 8192, 16)),
    ((32, 4096, 8192, 1), (33, 4096, 8192, 1)),
    ((33, 250, 8000, 1), (33, 250, 8192, 1)),
])
def test_rule(ring, tiles):
    assert plan(*ring) == RING
    assert plan(*tiles) != RING


# a batched score product: thousands of workgroups of one short stage each ran 4.6x longer on the ring
@pytest.mark.parametrize("m,n,k,batch", [(64, 4096, 64, 256), (33, 1000, 64, 64), (17, 512, 128, 64), (64, 512, 64, 1)])
def test_short_products_run_on_tiles(m, n, k, batch):
    assert plan(m, n, k, batch).startswith("gemm16_mfma_") or plan(m, n, k, batch).startswith("gemm16_dma_")
