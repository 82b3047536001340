"""float32 products on the 64x64 sequential-order ring (gemm_seq_ring.hip):
bit-identical to the oracle's fused-multiply-add recurrence in k order, around
its 16-k stages, its four-stage depth and its tile edges, in every operand
layout, with 16-byte rows and with rows of any length."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from tests.gemm_cases import assert_bit_exact, oracle_mm, randn
from torchvulkan_amd import _abi

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (63, 65, 15), (64, 64, 16), (65, 63, 17), (64, 128, 48), (68, 60, 64),
                                   (40, 100, 80), (130, 70, 333), (4, 200, 1)])
@pytest.mark.parametrize("pad", [0, 4, 3])
def test_bits(gpu, layout, m, n, k, pad):
    # rows `pad` elements wider than the operand, the rest NaN; a negative zero product keeps its sign rules too
    def wide(rows, cols, seed):
        t = torch.full((rows, cols + pad), float("nan"))
        t[:, :cols] = randn((rows, cols), torch.float32, seed)
        if cols > 2:
            t[0, :2] = torch.tensor([0.0, -0.0])
        return t.to(DEV)[:, :cols]

    a = wide(k, m, 1).t() if layout[0] == "t" else wide(m, k, 1)
    b = wide(n, k, 2).t() if layout[1] == "t" else wide(k, n, 2)
    c = torch.full((m, n), 7.0, device=DEV)
    assert gpu.gemm_plan(a, b, c) == "gemm_seq_mfma_64x64"
    _abi.gemm(a, b, c)
    torch.cuda.synchronize()
    assert_bit_exact(c.cpu().numpy(), oracle_mm(a.cpu(), b.cpu(), torch.float32).astype(np.float32), f"{layout} {m}x{n}x{k}")
