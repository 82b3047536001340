"""Kernel families of grad weights of odd planes: where the ring kernel's
channels-last copies would not fit its 2 GiB buffers, and where there are too
few output pixels for it (no GPU: the descriptors are not run)."""
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


# output pixels at and below its lines of 192 (up to 128 output channels) and 512
@pytest.mark.parametrize("batch,hw,kernel,stride,cin,cout,ring", [
    (1, 14, 3, 1, 64, 128, True), (3, 14, 3, 2, 64, 128, False), (1, 7, 3, 1, 512, 512, False), (1, 7, 1, 1, 8, 64, False),
    (12, 7, 3, 2, 64, 64, True), (11, 7, 3, 2, 64, 64, False),      # 192 and 176 pixels
    (1, 14, 3, 1, 64, 136, False), (2, 14, 3, 1, 256, 256, False),
    (32, 7, 3, 2, 256, 256, True), (31, 7, 3, 2, 256, 256, False),   # 512 and 496 pixels
])
def test_few_output_pixels(batch, hw, kernel, stride, cin, cout, ring):
    d = _abi.make_convnd_desc((batch, cin, hw, hw), (cout, cin, kernel, kernel), torch.float16, stride=stride,
                              padding=kernel // 2)
    d.x = d.weight = d.y = 256
    assert ("conv_ring" in _abi.conv_candidates(d, _abi.TVK_CONV_WGRAD)) == ring


# the copies' launch holds at most 2^24 workgroups (2^32 threads): batches of tiny planes past it
@pytest.mark.parametrize("batch,hw,kernel,ring", [(1 << 20, 1, 1, True), (1 << 23, 1, 1, False), (1 << 25, 1, 1, False),
                                                  ((1 << 22) - 1, 3, 3, True), (1 << 23, 3, 3, False)])
def test_more_workgroups_than_a_launch_holds(batch, hw, kernel, ring):
    d = _abi.make_convnd_desc((batch, 8, hw, hw), (8, 8, kernel, kernel), torch.float16, stride=1, padding=kernel // 2)
    d.x = d.weight = d.y = 256
    assert ("conv_ring" in _abi.conv_candidates(d, _abi.TVK_CONV_WGRAD)) == ring
