"""Kernel families of grad weights whose channels-last copies would not fit
the ring kernel's 2 GiB buffers (no GPU: the descriptors are not run)."""
from __future__ import annotations

import pytest
import torch

from torchvulkan_amd import _abi


# x of 7 x 7 planes is 1.5 times as large with the border of a 3x3 kernel: below, at and past 2 GiB of it
@pytest.mark.parametrize("batch,ring", [(1000, True), (25890, True), (25891, False), (40000, False)])
def test_bordered_copy_past_2_gib(batch, ring):
    d = _abi.make_convnd_desc((batch, 512, 7, 7), (64, 512, 3, 3), torch.float16, stride=1, padding=1)
    d.x = d.weight = d.y = 256   # 16-byte aligned, never dereferenced here
    assert (batch * 512 * 9 * 9 * 2 < 2**31) == ring and batch * 512 * 49 < 2**30
    names = _abi.conv_candidates(d, _abi.TVK_CONV_WGRAD)
    assert names == ["conv_ring", "conv_implicit_gemm"] if ring else names == ["conv_implicit_gemm"]
