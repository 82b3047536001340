"""The MFMA attention kernels at head dims other than 64 and 128: any multiple
of 8 up to 128, padded to tiles of 32, 64, 96 or 128 columns. Both directions
against the float64 oracle at the attention tests' tolerance (5e-3*(|ref|+1),
one bfloat16 step on at most 1 % of the elements), over the edges of each tile
width, ragged lengths around the 64-key tiles, and operands whose padding
columns hold NaN (nothing past the head dim may be read into a product)."""
from __future__ import annotations

import pytest
import torch

from oracle import oracle as orc
from tests.gemm_cases import assert_close
from tests.test_attention_gpu import DEV, check, check_bwd, f64, rand

pytestmark = pytest.mark.gpu


# smallest, one chunk below / at / above each tile width, largest
@pytest.mark.parametrize("dim", [8, 24, 32, 40, 56, 72, 80, 96, 104, 120])
@pytest.mark.parametrize("causal", [False, True])
def test_head_dims(gpu, dim, causal):
    dtype = torch.float16 if dim % 16 else torch.bfloat16
    q = rand((2, 4, 130, dim), dtype, dim)
    k, v = rand((2, 2, 130, dim), dtype, dim + 1), rand((2, 2, 130, dim), dtype, dim + 2)
    check(q, k, v, causal=causal, what=f"D {dim}")
    check_bwd(q, k, v, causal=causal, what=f"D {dim}")


@pytest.mark.parametrize("dim", [32, 80, 104])
@pytest.mark.parametrize("lens", [(1, 1), (63, 65), (64, 64), (65, 127), (3, 200)])
def test_lengths_and_bias(gpu, dim, lens):
    dtype = torch.float16
    n, s = lens
    q, k, v = rand((1, 3, n, dim), dtype, 7), rand((1, 3, s, dim), dtype, 8), rand((1, 3, s, dim), dtype, 9)
    bias = rand((1, 3, n, s), dtype, 10)
    if n > 2:
        bias[0, :, 2] = float("-inf")   # a row that attends to nothing
    check(q, k, v, bias=bias, what=f"D {dim} L {n} S {s}")
    check_bwd(q, k, v, bias=bias, what=f"D {dim} L {n} S {s}")
    check(q, k, v, causal=True, scale=-0.2, what=f"D {dim} L {n} S {s} causal")


@pytest.mark.parametrize("dim", [24, 80])
def test_columns_past_the_head_dim_are_not_used(gpu, dim):
    # views of wider rows whose further columns are NaN, head-strided underneath
    dtype = torch.float16

    def view(heads, n, seed):
        t = torch.full((1, n, heads, dim + 8), float("nan"), dtype=dtype)
        t[..., :dim] = rand((1, n, heads, dim), dtype, seed)
        return t.to(DEV)[..., :dim].transpose(1, 2)

    from torchvulkan_amd import _abi

    q, k, v, do = view(4, 70, 1), view(2, 70, 2), view(2, 70, 3), view(4, 70, 4)
    out, lse = _abi.attention_fwd(q, k, v, None, True)
    grads = _abi.attention_bwd(q, k, v, out, lse, do, None, True)
    torch.cuda.synchronize()
    ro, _ = orc.attention(f64(q), f64(k), f64(v), None, True)
    assert_close(f64(out), ro, dtype, "out")
    ref = orc.attention_bwd(f64(q), f64(k), f64(v), f64(do), None, True, None, out=f64(out), round_to=orc.F16)
    for got, want, name in zip(grads, ref, ("dq", "dk", "dv")):
        assert_close(f64(got), want, dtype, name)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("dim", [32, 64, 80, 128])
def test_masks_of_the_lowest_value(gpu, dtype, dim):
    # additive masks of the dtype's lowest finite value: masked keys get no weight beside an unmasked one, and a
    # row masked everywhere averages over its keys (the scores vanish beside the mask)
    low = torch.finfo(dtype).min
    q, k, v = rand((1, 2, 40, dim), dtype, 1), rand((1, 2, 70, dim), dtype, 2), rand((1, 2, 70, dim), dtype, 3)
    bias = torch.zeros((1, 2, 40, 70), dtype=dtype)
    bias[..., 50:] = low
    bias[:, :, 3, 1:] = low
    if dtype == torch.bfloat16:
        bias[:, :, 5] = low   # in float16 the scores do not vanish beside 65504, and the row is an ordinary one
    check(q, k, v, bias=bias, what=f"{dtype} D {dim}")


# the 128-query kernel with K and V loaded straight into LDS: the smallest grids that take it, lengths around its
# query blocks and key tiles, both LDS row widths, sliced keys whose further rows and columns are NaN
@pytest.mark.parametrize("dim,batch,heads", [(128, 16, 32), (104, 16, 32), (80, 16, 32), (64, 32, 32), (40, 32, 32)])
@pytest.mark.parametrize("lens,causal", [((127, 127), True), ((128, 64), False), ((100, 65), False), ((70, 200), True)])
def test_wide_kernel(gpu, dim, batch, heads, lens, causal):
    from torchvulkan_amd import _abi

    dtype = torch.float16 if dim % 16 else torch.bfloat16
    n, s = lens
    q = rand((batch, n, heads, dim), dtype, 1).to(DEV).transpose(1, 2)
    base = torch.full((batch, s + 9, 2, dim + 8), float("nan"), dtype=dtype)
    base[:, :s, :, :dim] = rand((batch, s, 2, dim), dtype, 2)
    kv = base.to(DEV)[:, :s, :, :dim].transpose(1, 2)
    out, lse = _abi.attention_fwd(q, kv, kv, None, causal, -0.1)
    torch.cuda.synchronize()
    for b, h in ((0, 0), (3, heads // 2), (batch - 1, heads - 1)):
        hk = h // (heads // 2)
        ro, rl = orc.attention(f64(q[b:b + 1, h:h + 1]), f64(kv[b:b + 1, hk:hk + 1]), f64(kv[b:b + 1, hk:hk + 1]), None,
                               causal, -0.1)
        assert_close(f64(out[b:b + 1, h:h + 1]), ro, dtype, f"b {b} h {h}")
        assert (abs(f64(lse[b:b + 1, h:h + 1]) - rl) <= 1e-3 * (abs(rl) + 1)).all()
    assert not out.isnan().any()


# the same kernel over several query blocks and key tiles (a tile's buffer is loaded again from the third on), heads
# and batches at both ends and in the middle; the last lengths have fewer queries than keys
@pytest.mark.parametrize("dim,batch,heads", [(128, 16, 32), (104, 16, 32), (80, 16, 32), (64, 16, 32)])
@pytest.mark.parametrize("lens,causal", [((300, 300), True), ((300, 300), False), ((200, 391), False), ((257, 449), True)])
def test_wide_kernel_over_many_tiles(gpu, dim, batch, heads, lens, causal):
    from tests.kernel_names import kernels
    from torchvulkan_amd import _abi

    dtype = torch.bfloat16 if dim % 16 else torch.float16
    n, s = lens
    q = rand((batch, n, heads, dim), dtype, 1).to(DEV).transpose(1, 2)
    k, v = (rand((batch, s, 2, dim), dtype, i).to(DEV).transpose(1, 2) for i in (2, 3))
    got = []
    names = kernels(lambda: got.append(_abi.attention_fwd(q, k, v, None, causal)))
    assert [x for x in names if "attn_fwd_wide_kernel" in x] == names and names, names
    out, lse = got[0]
    for b, h in ((0, 0), (batch // 2, heads // 2), (batch - 1, heads - 1)):
        hk = h // (heads // 2)
        ro, rl = orc.attention(f64(q[b:b + 1, h:h + 1]), f64(k[b:b + 1, hk:hk + 1]), f64(v[b:b + 1, hk:hk + 1]), None, causal)
        assert_close(f64(out[b:b + 1, h:h + 1]), ro, dtype, f"b {b} h {h}")
        assert (abs(f64(lse[b:b + 1, h:h + 1]) - rl) <= 1e-3 * (abs(rl) + 1)).all()


# heads, queries, dim, wide: both sides of the rule between the two forwards
@pytest.mark.parametrize("batch,heads,n,dim,wide", [
    (16, 32, 64, 128, False), (16, 32, 65, 128, True), (64, 32, 64, 104, False),
    (7, 73, 128, 96, False), (16, 16, 129, 80, True),      # 511 and 512 workgroups of 128 queries
    (32, 32, 64, 64, False), (32, 32, 65, 64, True), (64, 32, 17, 64, True), (89, 23, 17, 64, False),
    (16, 32, 192, 64, False), (16, 32, 193, 64, True), (16, 32, 192, 40, False), (16, 32, 193, 40, True),
])
def test_wide_dispatch(gpu, batch, heads, n, dim, wide):
    from tests.kernel_names import kernels
    from torchvulkan_amd import _abi

    q = torch.ones((batch, heads, n, dim), dtype=torch.float16, device=DEV)
    names = kernels(lambda: _abi.attention_fwd(q, q, q, None, True))
    assert all(("wide" in x) == wide for x in names) and names, names


def test_two_query_columns_with_a_bias(gpu):
    # head dim 64 with a bias on 2048 workgroups of 128 queries: the 64-query kernel's two-column form
    from tests.kernel_names import kernels
    from torchvulkan_amd import _abi

    dtype, batch, heads, n, s = torch.float16, 32, 32, 200, 130
    q, k, v = rand((batch, heads, n, 64), dtype, 1), rand((batch, 4, s, 64), dtype, 2), rand((batch, 4, s, 64), dtype, 3)
    bias = rand((1, heads, 1, s), dtype, 4)
    bias[..., 100:] = float("-inf")
    for causal in (False, True):
        got = []
        qd, kd, vd, bd = (t.to(DEV) for t in (q, k, v, bias))
        names = kernels(lambda: got.append(_abi.attention_fwd(qd, kd, vd, bd, causal)))
        assert len(names) == 1 and "attn_fwd_kernel" in names[0], names
        for b, h in ((0, 0), (13, 17), (31, 31)):
            hk = h // 8
            ro, rl = orc.attention(f64(q[b:b + 1, h:h + 1]), f64(k[b:b + 1, hk:hk + 1]), f64(v[b:b + 1, hk:hk + 1]),
                                   f64(bias[:, h:h + 1].expand(1, 1, n, s)), causal)
            assert_close(f64(got[0][0][b:b + 1, h:h + 1]), ro, dtype, f"b {b} h {h} causal {causal}")
            assert (abs(f64(got[0][1][b:b + 1, h:h + 1]) - rl) <= 1e-3 * (abs(rl) + 1)).all()
