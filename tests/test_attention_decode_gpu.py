"""Attention over a key/value cache (at most 16 queries, no causal mask): the
packed, key-split kernel of attention_decode.hip against the float64 oracle at
the attention tests' tolerance, at the edges of its 32-key tiles, 16-column row
blocks and splits, on sliced caches, with masks, and bit-identical when
repeated. A captured call (one split, no scratch) is replayed against it."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import oracle as orc
from tests.kernel_names import kernels
from tests.test_attention_gpu import DEV, assert_close, check, f64, rand
from torchvulkan_amd import _abi

pytestmark = pytest.mark.gpu


# keys: one, around a tile, around a wave's and a workgroup's share, several splits with a ragged end
@pytest.mark.parametrize("keys", [1, 31, 32, 33, 127, 129, 256, 1000, 2113])
@pytest.mark.parametrize("dim", [64, 128])
def test_keys(gpu, keys, dim):
    dtype = torch.bfloat16 if keys % 2 else torch.float16
    q, k, v = rand((2, 8, 1, dim), dtype, keys), rand((2, 2, keys, dim), dtype, keys + 1), rand((2, 2, keys, dim), dtype, 3)
    check(q, k, v, what=f"S {keys} D {dim}")
    check(q, k, v, scale=-0.3, what=f"S {keys} D {dim} negative scale")


# rows of one key/value head: 1, 15, 16, 17, 32, 33 and the largest, over one or two column blocks
@pytest.mark.parametrize("heads,new", [((1, 1), 1), ((3, 1), 5), ((8, 1), 2), ((17, 1), 1), ((4, 2), 16), ((33, 1), 1),
                                       ((8, 1), 16)])
@pytest.mark.parametrize("dim", [32, 80, 128])
def test_rows(gpu, heads, new, dim):
    dtype = torch.float16
    q = rand((2, heads[0], new, dim), dtype, 1)
    k, v = rand((2, heads[1], 700, dim), dtype, 2), rand((2, heads[1], 700, dim), dtype, 3)
    check(q, k, v, what=f"heads {heads} new {new} D {dim}")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("value", ["-inf", "lowest"])
def test_padding_masks(gpu, dtype, value):
    # a batch of different lengths: whole tiles, waves and splits are masked, and one sequence everywhere
    n, s = 2, 900
    low = float("-inf") if value == "-inf" else torch.finfo(dtype).min
    q, k, v = rand((3, 4, n, 64), dtype, 1), rand((3, 2, s, 64), dtype, 2), rand((3, 2, s, 64), dtype, 3)
    mask = torch.zeros((3, 1, 1, s), dtype=dtype)
    mask[0, ..., 5:] = low
    mask[1, ..., 640:] = low
    if value == "-inf":
        mask[2] = low
    check(q, k, v, bias=mask, what=f"{dtype} {value}")
    check(q, k, v, bias=rand((3, 4, n, s), dtype, 4), what=f"{dtype} dense bias")


@pytest.mark.parametrize("dim", [80, 128])
def test_sliced_cache_and_repeats(gpu, dim):
    # the filled part of a larger cache in [B, S, H, D] order; past it and past the head dim NaN
    dtype = torch.float16
    base = torch.full((2, 1100, 2, dim + 8), float("nan"), dtype=dtype)
    base[:, :1027, :, :dim] = rand((2, 1027, 2, dim), dtype, 5)
    kv = base.to(DEV)[:, :1027, :, :dim].transpose(1, 2)
    q = rand((2, 3, 8, dim), dtype, 6).to(DEV).transpose(1, 2)
    first = [t.clone() for t in _abi.attention_fwd(q, kv, kv)]
    for _ in range(3):
        out, lse = _abi.attention_fwd(q, kv, kv)
        torch.cuda.synchronize()
        assert torch.equal(out, first[0]) and torch.equal(lse, first[1])
    ro, rl = orc.attention(f64(q), f64(kv), f64(kv), None, False)
    assert_close(f64(first[0]), ro, dtype, "out")
    assert np.allclose(f64(first[1]), rl, rtol=1e-3, atol=1e-3)


def test_two_streams_and_capture(gpu):
    # concurrent calls keep their partials apart, and a captured call takes no scratch
    dtype = torch.float16
    q = [rand((2, 8, 1, 128), dtype, i).to(DEV) for i in range(2)]
    kv = [rand((2, 2, 4000, 128), dtype, 5 + i).to(DEV) for i in range(2)]
    want = [_abi.attention_fwd(q[i], kv[i], kv[i]) for i in range(2)]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(2)]
    got = [[], []]
    for _ in range(10):
        for i, st in enumerate(streams):
            with torch.cuda.stream(st):
                got[i].append(_abi.attention_fwd(q[i], kv[i], kv[i]))
    torch.cuda.synchronize()
    for i in range(2):
        for out, lse in got[i]:
            assert torch.equal(out, want[i][0]) and torch.equal(lse, want[i][1])
    out, lse = torch.empty_like(want[0][0]), torch.empty_like(want[0][1])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        d = _abi.make_attention_desc(q[0], kv[0], kv[0], out, lse, stream=torch.cuda.current_stream().cuda_stream)
        _abi.check(_abi.load().tvk_attention_fwd(d))
    for _ in range(3):
        out.zero_()
        graph.replay()
        again = _abi.attention_fwd(q[0], kv[0], kv[0])
        torch.cuda.synchronize()
        assert torch.equal(again[0], want[0][0])
        # one split instead of several: the same products merged in another order
        assert_close(f64(out), f64(want[0][0]), dtype, "captured")
        assert torch.allclose(lse, want[0][1], rtol=1e-5, atol=1e-5)


# infinities and NaN in V: a column that holds one is that value (or NaN) in every row that attends to it, the other
# columns are what they are without it. 3, 11 and 8 splits of the keys (the merge works on groups of eight), the value
# in the first, a middle and the last split; 1 and 40 query rows of a key/value head
@pytest.mark.parametrize("batch,heads,new,keys", [(2, (16, 16), 1, 700), (1, (8, 1), 1, 1400), (1, (8, 8), 5, 1000),
                                                  (2, (16, 2), 5, 1400), (1, (40, 1), 1, 1024)])
@pytest.mark.parametrize("dim", [64, 80, 128])
def test_non_finite_values(gpu, batch, heads, new, keys, dim):
    dtype = torch.bfloat16
    q, k = rand((batch, heads[0], new, dim), dtype, 1) * 0.1, rand((batch, heads[1], keys, dim), dtype, 2) * 0.1
    v = rand((batch, heads[1], keys, dim), dtype, 3)
    # (weights are all about 1 / keys: no product of a zero weight)
    for at, col, value in ((1, 3, float("inf")), (keys // 2, 17, float("-inf")), (keys - 1, 30, float("inf")),
                           (keys - 2, 31, float("nan"))):
        v[:, :, at, col] = value
    out, lse = _abi.attention_fwd(q.to(DEV), k.to(DEV), v.to(DEV))
    torch.cuda.synchronize()
    out = f64(out)
    assert (out[..., 3] == np.inf).all() and (out[..., 17] == -np.inf).all() and (out[..., 30] == np.inf).all()
    assert np.isnan(out[..., 31]).all()
    finite = [c for c in range(dim) if c not in (3, 17, 30, 31)]
    ro, rl = orc.attention(f64(q), f64(k), f64(torch.nan_to_num(v, 0.0, 0.0, 0.0)), None, False)
    assert_close(out[..., finite], ro[..., finite], dtype, "finite columns")
    assert np.allclose(f64(lse), rl, rtol=1e-3, atol=1e-3)


# batch, (heads), queries, keys, dim, mask, packed: both sides of the lines between this kernel and the tiled forward
@pytest.mark.parametrize("batch,heads,new,keys,dim,mask,packed", [
    (1, (8, 8), 16, 64, 128, False, False), (1, (8, 8), 16, 65, 128, False, True),       # a head's own keys: one tile
    (2, (16, 4), 4, 33, 128, False, True), (2, (16, 4), 5, 33, 128, False, False),       # 16 and 20 rows
    (1, (16, 4), 16, 512, 128, False, False), (1, (16, 4), 16, 513, 128, False, True),
    (1, (16, 4), 5, 448, 128, False, False), (1, (16, 4), 5, 449, 128, False, True),
    (2, (32, 1), 1, 384, 64, False, False), (2, (32, 1), 1, 385, 64, False, True),
    (2, (32, 1), 1, 384, 80, False, False), (2, (32, 1), 1, 385, 96, False, True),
    (8, (32, 8), 5, 300, 128, False, False), (9, (32, 8), 5, 300, 128, False, True),   # a round of heads
    (16, (32, 8), 5, 64, 128, False, False), (17, (32, 8), 5, 64, 128, False, True),
    (32, (32, 8), 16, 64, 64, False, False), (33, (32, 8), 16, 64, 64, False, True),
    (8, (32, 8), 16, 64, 128, True, False), (8, (32, 8), 16, 65, 128, True, True), (9, (32, 8), 16, 64, 64, True, True),
])
def test_dispatch(gpu, batch, heads, new, keys, dim, mask, packed):
    dtype = torch.float16
    q, k, v = (rand((batch, h, n, dim), dtype, i) for i, (h, n) in enumerate(((heads[0], new), (heads[1], keys), (heads[1], keys))))
    bias = rand((batch, 1, 1, keys), dtype, 4) if mask else None
    qd, kd, vd, bd = (None if t is None else t.to(DEV) for t in (q, k, v, bias))
    names = kernels(lambda: _abi.attention_fwd(qd, kd, vd, bd))
    assert any("attn_decode_kernel" in n for n in names) == packed and any("attn_fwd" in n for n in names) != packed, names
    check(q[:1], k[:1], v[:1], bias=None if bias is None else bias[:1], what="first batch")
