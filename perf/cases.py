"""The workloads whose speed this library is held to.

Each case is work that a program has the library do, called the way a program
calls it: serving loops and operator layers hold descriptors and call the C
ABI (tvk_gemm, tvk_conv_*, tvk_attention_*) on the current stream; training
programs run torch operators and autograd on the "vulkan" device.

Families (the "kind" of a case) and what they stand for:
  linear         nn.Linear in a serving step: few rows, weight [out, in]
  linear_train   nn.Linear with bias, forward and backward, on the vulkan device
  mm             a plain matrix product in one of its three layouts
  baddbmm        batched products with a batched bias, alpha and beta
  conv           a convolution layer: forward, grad input and grad weight
  sdpa_train     attention in a training step: forward and backward
  sdpa_prefill   attention over a prompt (forward only)
  sdpa_decode    attention of newly generated tokens over a key/value cache
  layer_step     a decoder layer's training step on the vulkan device
"""
from __future__ import annotations

import ctypes
import math

import torch

from torchvulkan_amd import _abi

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # the smallest call: a few tokens through a narrow projection, where latency and the launch count
        {"name": "linear_small", "kind": "linear", "dtype": "fp16", "tokens": 7, "fin": 512, "fout": 512, "bias": True},
        # decode through a wide up projection: the weight is read once and bounds the call
        {"name": "linear_decode", "kind": "linear", "dtype": "bf16", "tokens": 16, "fin": 4096, "fout": 14336,
         "bias": False},
        # ragged features and batch, as tabular and multimodal inputs have them, forward and backward
        {"name": "linear_train_ragged", "kind": "linear_train", "dtype": "fp16", "tokens": 1000, "fin": 777,
         "fout": 3000},
        # the largest call: a square half-precision product
        {"name": "mm_square", "kind": "mm", "dtype": "fp16", "layout": "nn", "m": 8192, "n": 8192, "k": 8192},
        # single precision, torch's default type
        {"name": "mm_fp32", "kind": "mm", "dtype": "fp32", "layout": "nn", "m": 1024, "n": 1024, "k": 1024},
        # small images: a strided stage of a residual network's training step
        {"name": "conv_small_image", "kind": "conv", "dtype": "fp16", "batch": 128, "cin": 64, "cout": 128, "hw": 32,
         "ksize": 3, "stride": 2, "bias": False, "dx": True},
        # photo-sized images: a middle stage, whose plane is no power of two
        {"name": "conv_photo", "kind": "conv", "dtype": "bf16", "batch": 32, "cin": 128, "cout": 128, "hw": 28,
         "ksize": 3, "stride": 1, "bias": False, "dx": True},
        # attention of a small decoder's training step, grouped key/value heads
        {"name": "sdpa_train", "kind": "sdpa_train", "dtype": "fp16", "batch": 32, "hq": 8, "hkv": 2, "len": 256,
         "dim": 64, "causal": True},
        # attention of an image encoder's training step: an odd token count, a head dimension that is no power of two
        {"name": "sdpa_train_image", "kind": "sdpa_train", "dtype": "bf16", "batch": 8, "hq": 16, "hkv": 16, "len": 577,
         "dim": 80, "causal": False},
        # attention over two prompts of odd length
        {"name": "sdpa_prefill", "kind": "sdpa_prefill", "dtype": "bf16", "batch": 2, "hq": 32, "hkv": 8, "len": 3001,
         "dim": 128, "causal": True},
        # one new token for each of eight sequences over a filled cache
        {"name": "sdpa_decode", "kind": "sdpa_decode", "dtype": "bf16", "batch": 8, "hq": 32, "hkv": 8, "new": 1,
         "len": 4001, "dim": 128, "mask": False},
        # a decoder layer's forward, loss and backward (grouped heads, gated feed-forward)
        {"name": "layer_step", "kind": "layer_step", "dtype": "fp16", "batch": 32, "len": 256, "hq": 8, "hkv": 2,
         "dim": 64, "ff": 1536},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi, grain=8, odd=0.3):
    """A size between lo and hi, spread over its logarithm: usually a multiple of `grain`, else any number."""
    v = _log_int(rng, lo, hi)
    return v if rng.random() < odd else max(lo, v // grain * grain)


def draw(rng):
    kind = rng.choice(["linear", "linear_train", "mm", "baddbmm", "conv", "sdpa_train", "sdpa_prefill", "sdpa_decode",
                       "layer_step"])
    half = rng.choice(["fp16", "bf16"])
    if kind == "linear":
        return {"kind": kind, "dtype": half, "tokens": _log_int(rng, 1, 64), "fin": _size(rng, 64, 8192, 64, 0.15),
                "fout": _size(rng, 64, 14336, 64, 0.15), "bias": rng.random() < 0.5}
    if kind == "linear_train":
        return {"kind": kind, "dtype": rng.choice(["fp16", "bf16", "fp32"]), "tokens": _size(rng, 16, 4096),
                "fin": _size(rng, 16, 2048), "fout": _size(rng, 8, 4096)}
    if kind == "mm":
        dtype = rng.choice(["fp16", "bf16", "fp32"])
        top = 2048 if dtype == "fp32" else 8000
        return {"kind": kind, "dtype": dtype, "layout": rng.choice(["nn", "nt", "tn"]), "m": _size(rng, 128, top, 64),
                "n": _size(rng, 128, top, 64), "k": _size(rng, 64, top, 64)}
    if kind == "baddbmm":
        return {"kind": kind, "dtype": half, "batch": _log_int(rng, 4, 256), "m": _size(rng, 16, 512, 16),
                "n": _size(rng, 16, 512, 16), "k": _size(rng, 16, 512, 16)}
    if kind == "conv":
        if rng.random() < 0.15:  # the first layer of a network: its input needs no gradient
            ksize, hw = rng.choice([(3, _size(rng, 28, 64, 4)), (7, _size(rng, 96, 224, 16))])
            return {"kind": kind, "dtype": half, "batch": _log_int(rng, 4, 64), "cin": 3,
                    "cout": rng.choice([16, 32, 48, 64]), "hw": hw, "ksize": ksize, "stride": 2 if ksize == 7 else 1,
                    "bias": rng.random() < 0.3, "dx": False}
        ksize, stride = rng.choice([(3, 1), (3, 1), (3, 2), (1, 1), (1, 2)])
        hw = rng.choice([7, 8, 14, 16, 27, 28, 32, 33, 56])
        cin = rng.choice([16, 32, 48, 64, 96, 128, 192, 256, 384, 512])
        cout = min(512, max(16, cin * rng.choice([1, 1, 2]) // rng.choice([1, 1, 2])))
        while hw * hw * max(cin, cout) > 256 * 1024:
            cin, cout = max(16, cin // 2), max(16, cout // 2)
        return {"kind": kind, "dtype": rng.choice([half, half, half, "fp32"]), "batch": _log_int(rng, 2, 64),
                "cin": cin, "cout": cout, "hw": hw, "ksize": ksize, "stride": stride, "bias": rng.random() < 0.3,
                "dx": True}
    group = rng.choice([1, 1, 2, 4, 8])
    hkv = rng.choice([1, 2, 4, 8])
    hq = min(32, hkv * group)
    dim = rng.choice([32, 64, 64, 80, 96, 128, 128])
    if kind == "sdpa_train":
        n = _size(rng, 32, 2048, 32)
        dtype = rng.choice(["fp16", "bf16", "fp16", "bf16", "fp32"])
        n = min(n, 512 if dtype == "fp32" else math.isqrt((1 << 26) // hq))
        batch = max(1, min(_log_int(rng, 1, 64), (1 << (22 if dtype == "fp32" else 26)) // (hq * n * n)))
        return {"kind": kind, "dtype": dtype, "batch": batch, "hq": hq, "hkv": hkv, "len": n, "dim": dim,
                "causal": rng.random() < 0.7}
    if kind == "sdpa_prefill":
        n = min(_size(rng, 128, 8192, 64), math.isqrt((1 << 28) // hq))
        batch = max(1, min(_log_int(rng, 1, 16), (1 << 28) // (hq * n * n)))
        return {"kind": kind, "dtype": half, "batch": batch, "hq": hq, "hkv": hkv, "len": n, "dim": dim,
                "causal": rng.random() < 0.8}
    if kind == "sdpa_decode":
        n = _size(rng, 32, 16384, 64, 0.6)
        batch = max(1, min(_log_int(rng, 1, 64), (1 << 28) // (hkv * n * dim)))
        return {"kind": kind, "dtype": half, "batch": batch, "hq": hq, "hkv": hkv, "new": rng.choice([1, 1, 1, 2, 5]),
                "len": n, "dim": dim, "mask": rng.random() < 0.3}
    n = _size(rng, 32, 1024, 32)
    batch = max(1, min(_log_int(rng, 4, 64), 8192 // n))
    hkv, hq = rng.choice([(1, 4), (2, 4), (2, 8), (4, 8), (8, 8), (12, 12)])
    return {"kind": kind, "dtype": half, "batch": batch, "len": n, "hq": hq, "hkv": hkv, "dim": rng.choice([32, 64]),
            "ff": _size(rng, 256, 2048, 64, 0.0)}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

class _Source:
    """Seeded normal values made on the GPU, rounded to the case's type."""

    def __init__(self, case, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed))
        self.dtype = DTYPES[case["dtype"]]

    def __call__(self, *shape, std=1.0, dtype=None):
        x = torch.randn(shape, generator=self.g, device="cuda", dtype=torch.float32)
        return (x * std if std != 1.0 else x).to(dtype or self.dtype)


def _conv_out(case):
    return (case["hw"] + 2 * (case["ksize"] // 2) - case["ksize"]) // case["stride"] + 1


def _inputs(case, seed):
    """The tensors of a case, on torch's own GPU device: what prepare() lays out and what exact() computes from."""
    r = _Source(case, seed)
    c = case
    kind = c["kind"]
    if kind == "linear":
        d = {"x": r(c["tokens"], c["fin"]), "w": r(c["fout"], c["fin"], std=c["fin"] ** -0.5)}
        if c["bias"]:
            d["b"] = r(c["fout"], std=0.1)
        return d
    if kind == "linear_train":
        return {"x": r(c["tokens"], c["fin"]), "w": r(c["fout"], c["fin"], std=c["fin"] ** -0.5),
                "b": r(c["fout"], std=0.1), "dy": r(c["tokens"], c["fout"])}
    if kind == "mm":
        a = r(c["k"], c["m"]).t() if c["layout"] == "tn" else r(c["m"], c["k"])
        b = r(c["n"], c["k"]).t() if c["layout"] == "nt" else r(c["k"], c["n"])
        return {"a": a, "b": b}
    if kind == "baddbmm":
        return {"a": r(c["batch"], c["m"], c["k"]), "b": r(c["batch"], c["k"], c["n"]),
                "c": r(c["batch"], c["m"], c["n"])}
    if kind == "conv":
        k, o = c["ksize"], _conv_out(c)
        d = {"x": r(c["batch"], c["cin"], c["hw"], c["hw"]),
             "w": r(c["cout"], c["cin"], k, k, std=(2.0 / (c["cin"] * k * k)) ** 0.5),
             "dy": r(c["batch"], c["cout"], o, o)}
        if c["bias"]:
            d["b"] = r(c["cout"], std=0.1)
        return d
    if kind in ("sdpa_train", "sdpa_prefill"):
        # [B, L, H, D] underneath: the projections' outputs split into heads
        def heads(h):
            return r(c["batch"], c["len"], h, c["dim"]).transpose(1, 2)

        d = {"q": heads(c["hq"]), "k": heads(c["hkv"]), "v": heads(c["hkv"])}
        if kind == "sdpa_train":
            d["do"] = heads(c["hq"])
        return d
    if kind == "sdpa_decode":
        cap = -(-c["len"] // 256) * 256  # the cache's capacity; the call sees its filled part
        d = {"q": r(c["batch"], c["new"], c["hq"], c["dim"]).transpose(1, 2),
             "k": r(c["batch"], c["hkv"], cap, c["dim"])[:, :, :c["len"]],
             "v": r(c["batch"], c["hkv"], cap, c["dim"])[:, :, :c["len"]]}
        if c["mask"]:  # sequences of different lengths in one batch: an additive mask over the padding
            g = torch.rand((c["batch"],), generator=r.g, device="cuda")
            fill = (c["len"] * (0.5 + 0.5 * g)).long().clamp(min=1)
            pad = torch.arange(c["len"], device="cuda")[None, :] >= fill[:, None]
            d["mask"] = torch.zeros(pad.shape, device="cuda", dtype=r.dtype).masked_fill_(pad, float("-inf"))
        return d
    width, dm = c["hq"] * c["dim"], c["hq"] * c["dim"]
    kv = c["hkv"] * c["dim"]
    t = c["batch"] * c["len"]

    def lin(fin, fout):
        return r(fout, fin, std=fin ** -0.5)

    return {"x": r(t, dm), "target": r(t, dm, dtype=torch.float32), "wq": lin(dm, width), "wk": lin(dm, kv),
            "wv": lin(dm, kv), "wo": lin(width, dm), "gate": lin(dm, c["ff"]), "up": lin(dm, c["ff"]),
            "down": lin(c["ff"], dm)}


# ---------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------

class _Calls:
    """Descriptors a program keeps over fixed buffers, and the buffers they write."""

    def __init__(self):
        self.calls, self.out, self.keep = [], {}, []

    def add(self, fn, desc):
        self.calls.append((getattr(_abi.load(), fn), ctypes.byref(desc)))
        self.keep.append(desc)

    def run(self):
        for fn, ref in self.calls:
            status = fn(ref)
            if status:
                _abi.check(status)
        return self.out


class _Vulkan:
    """Tensors on the vulkan device and the step a training program runs over them."""

    def __init__(self, case, tensors, step):
        self.case, self.t, self.step = case, tensors, step

    def run(self):
        return self.step(self.case, self.t)


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _to_vulkan(tensors, plain=()):
    got = {}
    for name, t in tensors.items():
        t = t.cpu().to("vulkan")
        got[name] = t if name in plain else t.requires_grad_()
    return got


def _grads(tensors):
    got = {}
    for name, t in tensors.items():
        if t.requires_grad:
            got["d_" + name] = t.grad
    return got


def _linear_train_step(case, t):
    for p in t.values():
        p.grad = None
    y = torch.nn.functional.linear(t["x"], t["w"], t["b"])
    y.backward(t["dy"])
    return {"y": y.detach(), **_grads(t)}


def _layer(c, t):
    f = torch.nn.functional
    bs, n = c["batch"], c["len"]
    q = f.linear(t["x"], t["wq"]).view(bs, n, c["hq"], c["dim"]).transpose(1, 2)
    k = f.linear(t["x"], t["wk"]).view(bs, n, c["hkv"], c["dim"]).transpose(1, 2)
    v = f.linear(t["x"], t["wv"]).view(bs, n, c["hkv"], c["dim"]).transpose(1, 2)
    a = f.scaled_dot_product_attention(q, k, v, is_causal=True, enable_gqa=True)
    h = t["x"] + f.linear(a.transpose(1, 2).reshape(bs * n, c["hq"] * c["dim"]), t["wo"])
    return h + f.linear(f.linear(h, t["gate"]) * f.linear(h, t["up"]), t["down"])


def _layer_step(case, t):
    for p in t.values():
        p.grad = None
    y = _layer(case, t)
    diff = y.float() - t["target"]
    loss = (diff * diff).sum()
    loss.backward()
    return {"loss": loss.detach(), "y": y.detach(), **_grads(t)}


def _conv_descs(case, t, s, got):
    pad = case["ksize"] // 2
    y = torch.empty_like(t["dy"])
    geometry = {"stride": case["stride"], "padding": pad, "stream": got}
    s.add("tvk_conv_fwd", _abi.conv_problem(t["x"], t["w"], y, bias=t.get("b"), **geometry))
    s.out["y"] = y
    if case["dx"]:
        dx = torch.empty_like(t["x"])
        s.add("tvk_conv_dgrad", _abi.conv_problem(dx, t["w"], t["dy"], **geometry))
        s.out["dx"] = dx
    dw = torch.empty_like(t["w"])
    s.add("tvk_conv_wgrad", _abi.conv_problem(t["x"], dw, t["dy"], **geometry))
    s.out["dw"] = dw


def _attention_descs(case, t, s, stream):
    q, k, v = t["q"], t["k"], t["v"]
    b, h, n, d = q.shape
    out = torch.empty((b, n, h, d), dtype=q.dtype, device=q.device).transpose(1, 2)  # the query's layout
    lse = torch.empty((b, h, n), dtype=torch.float32, device=q.device)
    mask = t["mask"][:, None, None, :] if "mask" in t else None
    fwd = _abi.make_attention_desc(q, k, v, out, lse, bias=mask, causal=bool(case.get("causal")), stream=stream)
    s.add("tvk_attention_fwd", fwd)
    s.out.update(out=out, lse=lse)
    if case["kind"] != "sdpa_train":
        return
    bwd = _abi.AttentionBwdDesc()
    bwd.fwd = fwd
    grads = {"dout": t["do"]}
    for name, like in (("dq", q), ("dk", k), ("dv", v)):
        grads[name] = s.out[name] = torch.empty(like.shape, dtype=like.dtype, device=like.device)
    for name, g in grads.items():
        setattr(bwd, name, g.data_ptr())
        setattr(bwd, name + "_stride", _abi.I64x4(*g.stride()))
    s.add("tvk_attention_bwd", bwd)


def prepare(case, seed):
    t = _inputs(case, seed)
    kind = case["kind"]
    if kind == "linear_train":
        return _Vulkan(case, _to_vulkan(t, plain=("dy",)), _linear_train_step)
    if kind == "layer_step":
        return _Vulkan(case, _to_vulkan(t, plain=("target",)), _layer_step)
    s, stream = _Calls(), _stream()
    s.keep.append(t)
    if kind == "conv":
        _conv_descs(case, t, s, stream)
    elif kind.startswith("sdpa"):
        _attention_descs(case, t, s, stream)
    else:
        more = {}
        if kind == "linear":
            a, b = t["x"], t["w"].t()
            if case["bias"]:
                more = {"bias": t["b"], "beta": 1.0}
        else:
            a, b = t["a"], t["b"]
            if kind == "baddbmm":
                more = {"bias": t["c"], "alpha": 0.5, "beta": 1.0}
        c = torch.empty((*a.shape[:-1], b.shape[-1]), dtype=a.dtype, device=a.device)
        s.add("tvk_gemm", _abi.make_gemm_desc(a, b, c, stream=stream, **more))
        s.out["c"] = c
    return s


def run(state):
    return state.run()


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def work(case):
    c = case
    e = 4 if c["dtype"] == "fp32" else 2
    kind = c["kind"]
    if kind == "linear":
        m, k, n = c["tokens"], c["fin"], c["fout"]
        return {"bytes": e * (m * k + k * n + m * n + (n if c["bias"] else 0)), "flops": 2 * m * n * k}
    if kind == "linear_train":
        m, k, n = c["tokens"], c["fin"], c["fout"]
        # forward x, w, b -> y; backward dy, w, x -> dx, dw, db
        return {"bytes": e * (3 * m * k + 3 * k * n + 2 * m * n + 2 * n), "flops": 6 * m * n * k}
    if kind in ("mm", "baddbmm"):
        batch, m, n, k = c.get("batch", 1), c["m"], c["n"], c["k"]
        outs = 2 if kind == "baddbmm" else 1
        return {"bytes": e * batch * (m * k + k * n + outs * m * n), "flops": 2 * batch * m * n * k}
    if kind == "conv":
        x = c["batch"] * c["cin"] * c["hw"] ** 2
        y = c["batch"] * c["cout"] * _conv_out(c) ** 2
        w = c["cout"] * c["cin"] * c["ksize"] ** 2
        passes = 3 if c["dx"] else 2
        return {"bytes": e * passes * (x + y + w) + (e * c["cout"] if c["bias"] else 0),
                "flops": 2 * passes * y * c["cin"] * c["ksize"] ** 2}
    if kind.startswith("sdpa"):
        n, rows = c["len"], c.get("new", c["len"])
        q = c["batch"] * c["hq"] * rows * c["dim"]
        kv = c["batch"] * c["hkv"] * n * c["dim"]
        scores = c["batch"] * c["hq"] * (n * (n + 1) // 2 if c.get("causal") else rows * n)
        lse = 4 * c["batch"] * c["hq"] * rows
        got = {"bytes": e * (2 * q + 2 * kv) + lse, "flops": 4 * scores * c["dim"]}
        if c.get("mask"):
            got["bytes"] += e * c["batch"] * n
        if kind == "sdpa_train":  # backward: q, k, v, out, dout, lse -> dq, dk, dv; five products
            got["bytes"] += e * (4 * q + 4 * kv) + lse
            got["flops"] += 10 * scores * c["dim"]
        return got
    t, dm, kv, ff = c["batch"] * c["len"], c["hq"] * c["dim"], c["hkv"] * c["dim"], c["ff"]
    weights = 2 * dm * dm + 2 * dm * kv + 3 * dm * ff
    scores = c["batch"] * c["hq"] * c["len"] * (c["len"] + 1) // 2
    # each product's input is kept for its backward; weights are read twice and their gradients written
    acts = t * (3 * dm + 2 * dm + 2 * kv + 3 * ff)
    return {"bytes": e * (3 * weights + 3 * acts) + 12 * t * dm, "flops": 6 * t * weights + 14 * scores * c["dim"]}


def tolerance(case):
    """Four times the error against 64 bits that correct rounding to the case's type shows: one rounding of each
    output in a single layer, a few of them in a row where the values between (probabilities, a layer's
    activations and gradients) are rounded too."""
    kind, dtype = case["kind"], case["dtype"]
    if dtype == "fp32":
        return {"rel": 4e-6}
    steps = 3.0 if kind == "layer_step" else 1.4 if kind.startswith("sdpa") else 1.0
    return {"rel": steps * (8.5e-4 if dtype == "fp16" else 7e-3)}


# ---------------------------------------------------------------------------
# the same outputs in 64 bits
# ---------------------------------------------------------------------------

def _exact_attention(q, k, v, causal, mask=None, do=None):
    """One batch entry in float64: q [Hq, L, D], k and v [Hkv, S, D], mask [S] or None; out, lse and, for a
    gradient do of out, the gradients of q, k and v."""
    q, k, v = q.double(), k.double(), v.double()
    heads, rep, scale = k.shape[0], q.shape[0] // k.shape[0], q.shape[-1] ** -0.5
    k, v = k.repeat_interleave(rep, 0), v.repeat_interleave(rep, 0)
    s = torch.matmul(q, k.transpose(1, 2).contiguous()) * scale
    if mask is not None:
        s += mask.double()
    if causal:
        s.masked_fill_(~torch.ones(s.shape[1:], dtype=torch.bool, device=s.device).tril(), float("-inf"))
    lse = torch.logsumexp(s, -1)
    p = s.sub_(lse[..., None]).exp_()
    out = torch.matmul(p, v)
    if do is None:
        return out, lse
    do = do.double()
    ds = torch.matmul(do, v.transpose(1, 2).contiguous()).sub_((do * out).sum(-1, keepdim=True)).mul_(p).mul_(scale)

    def per_head(x):  # a key/value head's gradient sums over the query heads that read it
        return x.view(heads, rep, *x.shape[1:]).sum(1)

    dk = per_head(torch.matmul(ds.transpose(1, 2).contiguous(), q))
    dv = per_head(torch.matmul(p.transpose(1, 2).contiguous(), do))
    return out, lse, torch.matmul(ds, k), dk, dv


def _exact_conv(case, t):
    """A convolution as one product per tap, in float64."""
    n, ci, hw, _ = t["x"].shape
    k, s, p, o = case["ksize"], case["stride"], case["ksize"] // 2, _conv_out(case)
    co = case["cout"]
    xp = torch.nn.functional.pad(t["x"].double(), (p, p, p, p))
    w, dy = t["w"].double(), t["dy"].double().reshape(n, co, o * o)
    y = torch.zeros((n, co, o * o), dtype=torch.float64, device=xp.device)
    dxp, dw = torch.zeros_like(xp), torch.empty_like(w)
    rows = dy.transpose(0, 1).reshape(co, n * o * o)
    for a in range(k):
        for b in range(k):
            at = (slice(None), slice(None), slice(a, a + s * (o - 1) + 1, s), slice(b, b + s * (o - 1) + 1, s))
            tap = w[:, :, a, b].contiguous()
            x = xp[at].reshape(n, ci, o * o)
            y += torch.matmul(tap, x)
            dw[:, :, a, b] = rows @ x.permute(0, 2, 1).reshape(n * o * o, ci)
            if case["dx"]:
                dxp[at] += torch.matmul(tap.t().contiguous(), dy).reshape(n, ci, o, o)
    y = y.reshape(n, co, o, o)
    if "b" in t:
        y += t["b"].double().view(1, co, 1, 1)
    got = {"y": y, "dw": dw}
    if case["dx"]:
        got["dx"] = dxp[:, :, p:p + hw, p:p + hw].contiguous()
    return got


def _exact_layer(case, t):
    t = {name: x.double() for name, x in t.items()}
    x, bs, n, dim = t["x"], case["batch"], case["len"], case["dim"]

    def split(y, h):
        return y.view(bs, n, h, dim).transpose(1, 2)

    def joined(parts):
        return torch.stack(parts).transpose(1, 2).reshape(bs * n, -1)

    q, k, v = (split(x @ t[w].t(), case[h]) for w, h in (("wq", "hq"), ("wk", "hkv"), ("wv", "hkv")))
    a = joined([_exact_attention(q[i], k[i], v[i], True)[0] for i in range(bs)])
    h = x + a @ t["wo"].t()
    g, u = h @ t["gate"].t(), h @ t["up"].t()
    m = g * u
    y = h + m @ t["down"].t()
    diff = y - t["target"]
    dy = 2 * diff
    dm = dy @ t["down"]
    dg, du = dm * u, dm * g
    dh = dy + dg @ t["gate"] + du @ t["up"]
    da = split(dh @ t["wo"], case["hq"])
    parts = [_exact_attention(q[i], k[i], v[i], True, None, da[i])[2:] for i in range(bs)]
    dq, dk, dv = (joined([p[i] for p in parts]) for i in range(3))
    return {"loss": (diff * diff).sum(), "y": y, "d_x": dh + dq @ t["wq"] + dk @ t["wk"] + dv @ t["wv"],
            "d_wq": dq.t() @ x, "d_wk": dk.t() @ x, "d_wv": dv.t() @ x, "d_wo": dh.t() @ a, "d_gate": dg.t() @ h,
            "d_up": du.t() @ h, "d_down": dy.t() @ m}


def exact(case, seed):
    t = _inputs(case, seed)
    kind = case["kind"]
    if kind == "linear":
        c = t["x"].double() @ t["w"].double().t()
        return {"c": c + t["b"].double() if case["bias"] else c}
    if kind == "linear_train":
        x, w, b, dy = (t[name].double() for name in ("x", "w", "b", "dy"))
        return {"y": x @ w.t() + b, "d_x": dy @ w, "d_w": dy.t() @ x, "d_b": dy.sum(0)}
    if kind == "mm":
        return {"c": t["a"].double() @ t["b"].double()}
    if kind == "baddbmm":
        return {"c": t["c"].double() + 0.5 * torch.matmul(t["a"].double(), t["b"].double())}
    if kind == "conv":
        return _exact_conv(case, t)
    if kind == "layer_step":
        return _exact_layer(case, t)
    names = ("out", "lse", "dq", "dk", "dv") if kind == "sdpa_train" else ("out", "lse")
    parts = [_exact_attention(t["q"][i], t["k"][i], t["v"][i], bool(case.get("causal")),
                              t["mask"][i] if "mask" in t else None, t["do"][i] if "do" in t else None)
             for i in range(case["batch"])]
    return {name: torch.stack([p[i] for p in parts]) for i, name in enumerate(names)}
