"""Performance cases: the passes and layers a user of this framework runs.

Each case is one pass through a public entry point: a whole network or a
layer through :class:`~quantanything_amd.executor.DeviceExecutor` (float
input already in HBM, the captured pass replayed, float outputs left in
HBM), a standalone device GEMM (``workloads.GemmWorkload``), or a layer of
host arrays through the reference's own calls (``native.py``). Networks are
the repository's seeded builders, calibrated once per process on fixed data;
a case's seed makes its input batch alone. Tiles are the library's own
choice, as in ``QuantContainer.run_graph``.
"""

import math
import os
import tempfile
from functools import lru_cache

import numpy as np
import torch

from quantanything_amd import graph as G
from quantanything_amd import native
from quantanything_amd.container import QuantContainer
from quantanything_amd.executor import DeviceExecutor
from quantanything_amd.synth import Stream
from quantanything_amd.workloads import GemmWorkload


# ------------------------------------------------------------------ cases --
def listed():
    return [
        # The classifier the framework is benchmarked on: a full batch, and
        # one image, where launches and latency are all there is.
        dict(name="cls_b64", kind="cls", type="int8", batch=64, size=224),
        dict(name="cls_b1", kind="cls", type="int8", batch=1, size=224),
        # The same network quantized to 16 bits.
        dict(name="cls_int16_b64", kind="cls", type="int16", batch=64,
             size=224),
        # ViT-S/16: weight GEMMs, attention, LayerNorm over 197 tokens.
        dict(name="vit_b32", kind="vit", type="int8", batch=32, size=224,
             dim=384, heads=6, depth=12),
        # A network with depthwise and pointwise convolutions, a C2f block
        # and a pool over a 56x56 map, at a mobile backbone's width.
        dict(name="mobile_b32", kind="mobile", type="int8", batch=32,
             size=224, width=32),
        # A detector's neck: chained MaxPools, Concat, Pad, a feature map
        # handed back as floats.
        dict(name="sppf_b16", kind="sppf", type="int8", batch=16, size=224,
             width=64),
        # One Conv -> SiLU layer between float feature maps (a model run
        # layer by layer, or a backbone's last layer), and a small one with
        # odd sizes.
        dict(name="conv_b32", kind="conv", type="int8", batch=32, cin=64,
             cout=64, size=56, k=3, stride=1),
        dict(name="conv_ragged", kind="conv", type="uint8", batch=5, cin=24,
             cout=40, size=57, k=3, stride=1),
        # Device-resident GEMMs with their requantize: a large linear layer
        # and the narrow one of the standalone benchmark.
        dict(name="gemm_large", kind="gemm", m=16384, k=1024, n=1024),
        dict(name="gemm_narrow", kind="gemm", m=4096, k=576, n=64),
        # A fully connected layer whose sizes are multiples of nothing
        # useful, between float matrices.
        dict(name="fc_ragged", kind="fc", type="int8", m=1000, k=500, n=250),
        # A Conv -> requantize -> table layer of host arrays, as the
        # reference's container calls the library it loads.
        dict(name="host_conv", kind="host", op="int", batch=8, cin=64,
             cout=64, size=56, k=3),
    ]


def _log(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi]."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(
        math.log(lo), math.log(hi)))))))


def _most(kind, rng_type):
    """Bounds of a drawn case's work: those of the kind's largest listed
    case (of its type, where types differ in cost)."""
    same = [c for c in listed() if c["kind"] == kind]
    typed = [c for c in same if c.get("type") == rng_type] or same
    w = [work(c) for c in typed]
    return max(v["bytes"] for v in w), max(v["flops"] for v in w)


def draw(rng):
    kind = rng.choice(["cls", "vit", "mobile", "sppf", "conv", "conv",
                       "gemm", "gemm", "fc", "host"])
    while True:
        c = dict(kind=kind)
        if kind == "cls":
            c.update(type=rng.choice(["int8", "uint8", "int16"]),
                     batch=_log(rng, 1, 64), size=rng.randint(96, 224))
        elif kind == "vit":
            heads = rng.choice([2, 3, 4, 6])
            c.update(type=rng.choice(["int8", "uint8"]),
                     batch=_log(rng, 1, 32), size=16 * rng.randint(4, 15),
                     dim=64 * heads, heads=heads, depth=rng.randint(1, 4))
        elif kind == "mobile":
            c.update(type=rng.choice(["int8", "uint8", "int16"]),
                     batch=_log(rng, 1, 32), size=rng.randint(64, 224),
                     width=_log(rng, 4, 32))
            if c["type"] == "int16":  # the 16-bit path costs more
                c.update(batch=min(c["batch"], 8), width=min(c["width"], 16))
        elif kind == "sppf":
            c.update(type=rng.choice(["int8", "uint8"]),
                     batch=_log(rng, 1, 16), size=rng.randint(64, 224),
                     width=2 * _log(rng, 4, 32))
        elif kind == "conv":
            c.update(type=rng.choice(["int8", "uint8", "int16"]),
                     batch=_log(rng, 1, 64), cin=_log(rng, 3, 512),
                     cout=_log(rng, 8, 512), size=_log(rng, 7, 112),
                     k=rng.choice([1, 3, 3, 5]), stride=rng.choice([1, 1, 2]))
            if c["type"] == "int16":
                c.update(batch=min(c["batch"], 8))
        elif kind == "gemm":  # rows of activations are 16-byte aligned
            c.update(m=_log(rng, 1, 16384), k=16 * _log(rng, 2, 256),
                     n=_log(rng, 16, 4096))
        elif kind == "fc":
            c.update(type=rng.choice(["int8", "uint8", "int16"]),
                     m=_log(rng, 1, 4096), k=_log(rng, 16, 1280),
                     n=_log(rng, 10, 1000))
        else:
            c.update(op=rng.choice(["int", "wide", "float"]),
                     batch=_log(rng, 1, 8), cin=_log(rng, 8, 128),
                     cout=_log(rng, 8, 128), size=_log(rng, 7, 56),
                     k=rng.choice([1, 3]))
        most, w = _most(kind, c.get("type")), work(c)
        # channel halves off the 16-byte grid take general kernels
        share = 40 if kind == "mobile" and c["width"] % 16 else 1
        if w["bytes"] <= most[0] and share * w["flops"] <= most[1]:
            return c


# --------------------------------------------------------------- networks --
def _graph(c, batch):
    """The case's graph and its input's name and shape."""
    kind = c["kind"]
    if kind == "fc":
        return G.gemm_layer(k=c["k"], n=c["n"]), "x", (batch, c["k"])
    if kind == "conv":
        return G.conv_silu(cin=c["cin"], cout=c["cout"], size=c["size"],
                           k=c["k"], stride=c["stride"]), "x", \
            (batch, c["cin"], c["size"], c["size"])
    shape = (batch, 3, c["size"], c["size"])
    if kind == "vit":
        g = G.vit(batch=batch, size=c["size"], dim=c["dim"],
                  depth=c["depth"], heads=c["heads"], mlp=4 * c["dim"])
    elif kind == "cls":
        g = G.yolov8n_cls(size=c["size"])
    elif kind == "mobile":
        g = G.mini_yolo(size=c["size"], width=c["width"])
    else:
        g = G.mini_sppf(size=c["size"], width=c["width"])
    if g.nodes[-1].op_type == "Softmax":  # the logits beside the classes
        g.outputs = [g.nodes[-1].inputs[0]] + g.outputs
    return g, "images", shape


@lru_cache(maxsize=1)
def _container(items):
    """The case's network, calibrated on two fixed images or 64 fixed rows
    (through its q.json, as a deployed model is loaded)."""
    c = dict(items)
    g, name, shape = _graph(c, 64 if c["kind"] == "fc" else 2)
    q = QuantContainer(g, c["type"], per_channel=True)
    q.calibrate([{name: Stream(77).normal(shape).astype(np.float32)}])
    with tempfile.TemporaryDirectory() as d:
        path = os.path.join(d, "q.json")
        q.save(path)
        return QuantContainer.load(_graph(c, c.get("batch", c.get("m")))[0],
                                   path)


def _key(case):
    return tuple(sorted((k, v) for k, v in case.items() if k != "name"))


def _normal(shape, seed):
    """The float input batch: N(0, 1), on the GPU."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(shape, generator=gen, device="cuda")


# ------------------------------------------------------------- host layer --
def _host_inputs(c, seed):
    """Centred integer activations and weights of one layer, as the
    reference's container holds them (or floats), its requantization
    parameters and table."""
    r = np.random.default_rng(seed)
    shape = (c["batch"], c["cin"], c["size"], c["size"])
    wshape = (c["cout"], c["cin"], c["k"], c["k"])
    if c["op"] == "float":
        return dict(x=r.standard_normal(shape, np.float32),
                    w=r.standard_normal(wshape, np.float32))
    lim = 32767 if c["op"] == "wide" else 127
    n = c["cin"] * c["k"] ** 2
    mult = r.integers(1 << 30, 1 << 31, c["cout"])
    # accumulators of about lim^2 / 3 * sqrt(n) to about half the range
    shift = int(round(math.log2(lim * math.sqrt(n) / 2)))
    out = np.arange(-lim - 1, lim + 1)
    return dict(
        x=r.integers(-lim - 1, lim + 1, shape).astype(np.int32),
        w=r.integers(-lim, lim + 1, wshape).astype(
            np.int32 if c["op"] == "wide" else np.int16),
        mult=mult, shift=np.full(c["cout"], shift),
        bias=r.integers(-4096, 4097, c["cout"]), lim=lim,
        lut=np.maximum(out, out >> 3).astype(np.int32))


def _geometry(c):
    p = c["k"] // 2
    return c["size"] + 2 * p - c["k"] + 1, (p, p, p, p)


# ------------------------------------------------------------------- pass --
def prepare(case, seed):
    kind = case["kind"]
    if kind == "gemm":
        return dict(gemm=GemmWorkload(seed=seed, M=case["m"], K=case["k"],
                                      N=case["n"]))
    if kind == "host":
        return dict(host=_host_inputs(case, seed), case=case)
    q = _container(_key(case))
    name, shape = _graph_input(case)
    ex = DeviceExecutor(q, {name: shape})
    ex.inputs_f32[name].copy_(_normal(shape, seed))
    ex.capture()
    return dict(ex=ex)


def _graph_input(case):
    if case["kind"] == "fc":
        return "x", (case["m"], case["k"])
    if case["kind"] == "conv":
        return "x", (case["batch"], case["cin"], case["size"], case["size"])
    return "images", (case["batch"], 3, case["size"], case["size"])


def run(state):
    if "ex" in state:
        state["ex"].replay()
        return state["ex"].outputs_f32
    if "gemm" in state:
        state["gemm"].launch()
        return state["gemm"].y
    c, h = state["case"], state["host"]
    o, pads = _geometry(c)
    if c["op"] == "float":
        return native.conv2d_f32(h["x"], h["w"], pads=pads)
    acc = native.conv2d_int(h["x"], h["w"], pads=pads, wide=c["op"] == "wide")
    q = native.requantize(acc, c["batch"], c["cout"], o * o, h["mult"],
                          h["shift"], 0, -h["lim"] - 1, h["lim"],
                          pre_bias=h["bias"])
    return native.lut(q, h["lut"], -h["lim"] - 1)


# ------------------------------------------------------------------- work --
def work(case):
    """Float input in, float outputs out, weights once; two operations a
    multiply-add of the network's convolutions and products."""
    k = case["kind"]
    if k == "gemm":
        m, kk, n = case["m"], case["k"], case["n"]
        return dict(bytes=m * kk + kk * n + m * n + 24 * n, flops=2 * m * kk * n)
    wb = 2 if case.get("type") == "int16" else 1
    if k == "fc":
        m, kk, n = case["m"], case["k"], case["n"]
        return dict(bytes=4 * m * kk + wb * kk * n + 4 * m * n,
                    flops=2 * m * kk * n)
    b, s = case["batch"], case["size"]
    if k == "host":
        o, _ = _geometry(case)
        x, w = b * case["cin"] * s * s, case["cout"] * case["cin"] * case["k"] ** 2
        y = b * case["cout"] * o * o
        return dict(bytes=4 * x + w * (2 if case["op"] == "int" else 4) + 4 * y,
                    flops=2 * y * case["cin"] * case["k"] ** 2)
    if k == "conv":
        o = (s + 2 * (case["k"] // 2) - case["k"]) // case["stride"] + 1
        w = case["cin"] * case["cout"] * case["k"] ** 2
        return dict(bytes=4 * b * case["cin"] * s * s + wb * w +
                    4 * b * case["cout"] * o * o, flops=2 * b * o * o * w)
    img = 4 * b * 3 * s * s
    if k == "cls":
        return dict(bytes=img + wb * 2.72e6 + 8000 * b,
                    flops=0.4052e9 * b * (s / 224) ** 2)
    if k == "vit":
        t, d, mlp = (s // 16) ** 2 + 1, case["dim"], 4 * case["dim"]
        wl = 4 * d * d + 2 * d * mlp
        wts = case["depth"] * wl + 768 * d + 1000 * d
        mac = case["depth"] * (t * wl + 2 * t * t * d) + (t - 1) * 768 * d + \
            1000 * d
        return dict(bytes=img + wts + 4000 * b, flops=2 * b * mac)
    s2, s4 = -(-s // 2), -(-(-(-s // 2)) // 2)
    if k == "mobile":
        w = case["width"]
        mac = s2 * s2 * 27 * w + s4 * s4 * (18 * w * w + 18 * w * w + 12 * w * w
                                            + 36 * w + 32 * w * w) + 80 * w
        return dict(bytes=img + wb * 80 * w * w + 80 * b, flops=2 * b * mac)
    w, c = case["width"], case["width"] // 2
    p4 = (s2 + 1) * (s2 + 1)
    mac = s2 * s2 * (27 * w + w * c + 4 * c * w) + p4 * 9 * (w + 3) * w
    return dict(bytes=img + 14 * w * w + 4 * b * w * s2 * s2 + 40 * b,
                flops=2 * b * mac)


def tolerance(case):
    """Integer results are the reference's, bit for bit; only the float
    fallbacks may differ, by a step where a sum is within rounding of a tie
    (a transformer's LayerNorm and activation products)."""
    if case["kind"] == "host" and case["op"] == "float":
        return {"rel": 1e-5}  # float32 sums in another order
    if case["kind"] == "vit":
        # (one in 10^8 of the variance moved, so that a few values of a layer
        # step, moves the logits of twelve layers by 1.7e-2)
        return {"rel": 3e-2}
    return "exact"


def exact(case, seed):
    """The layer in 64 bits; None for the networks, whose result is the
    quantized one by definition."""
    k = case["kind"]
    if k == "gemm":
        g = GemmWorkload(seed=seed, M=case["m"], K=case["k"], N=case["n"]).spec
        a = torch.from_numpy(g["a"]).cuda().double() - g["zp_in"]
        acc = (a @ torch.from_numpy(g["w"]).cuda().double()).long()
        t = torch.from_numpy(31 + g["shift"]).cuda()
        v = (acc + torch.from_numpy(g["bias"]).cuda()) * \
            torch.from_numpy(g["mult"]).cuda()
        q = (v + (torch.ones_like(t) << (t - 1))) >> t
        q = (q + g["zp_out"]).clamp(g["qmin"], g["qmax"])
        return (q - 128).to(torch.int8).reshape(-1)
    if k == "host":
        h = _host_inputs(case, seed)
        o, pads = _geometry(case)
        acc = torch.nn.functional.conv2d(
            torch.from_numpy(h["x"]).double(),
            torch.from_numpy(h["w"].astype(np.float64)), padding=pads[0])
        if case["op"] == "float":
            return acc
        # accumulators are below 2^53; their products with the multipliers,
        # up to 2^72, are taken in two parts
        acc = acc.numpy().astype(np.int64) + h["bias"].reshape(1, -1, 1, 1)
        m = h["mult"].reshape(1, -1, 1, 1)
        t = 31 + int(h["shift"][0])
        low = ((acc & 0xFFFF) * m + (1 << (t - 1))) >> 16
        q = ((acc >> 16) * m + low) >> (t - 16)
        q = np.clip(q, -h["lim"] - 1, h["lim"])
        return h["lut"][q + h["lim"] + 1]
    if k not in ("conv", "fc"):
        return None
    g = _graph(case, case.get("batch", case.get("m")))[0]
    init = {n: torch.from_numpy(v).double() for n, v in
            g.initializers.items() if v.dtype == np.float32}
    x = _normal(_graph_input(case)[1], seed).cpu().double()
    w, b = (init[n] for n in g.nodes[0].inputs[1:])
    if k == "fc":
        y = x @ w + b
    else:
        y = torch.nn.functional.silu(torch.nn.functional.conv2d(
            x, w, b, stride=case["stride"], padding=case["k"] // 2))
    return {g.outputs[0]: y}
