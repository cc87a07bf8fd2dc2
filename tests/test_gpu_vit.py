"""Transformer operators on the GPU vs the oracle pipeline: the float
fallbacks of the integer pass (LayerNorm, activation x activation MatMul,
Softmax over the last axis of 4-D tensors, Gather; ``quant_layers.py:195-205``)
agree within one quantization step of the oracle on the same input, and
every integer layer around them (weight MatMuls with fused bias / Gelu
table / residual Add, layout views, token Concat, broadcast position Add) is
bit-exact given the same inputs (the oracle is run with the device's
fallback outputs substituted for its own)."""

import numpy as np
import pytest

from oracle.pipeline import OraclePipeline
from quantanything_amd import graph as G
from quantanything_amd.container import QuantContainer
from quantanything_amd.synth import Stream

pytestmark = pytest.mark.gpu

FALLBACK_OPS = ("LayerNormalization", "Softmax", "Gather")


def _calibrated(g, quant_type, batches):
    c = QuantContainer(g, quant_type, True)
    c.calibrate(batches)
    return c


def _fallback_outputs(g):
    return [n.outputs[0] for n in g.nodes if n.op_type in FALLBACK_OPS or (
        n.op_type == "MatMul" and n.inputs[1] not in g.initializers)]


def _check_against_oracle(c, g, tmp_path, x, ex, name="images"):
    """Runs the oracle with the device's fallback outputs; returns the worst
    fallback difference (steps) and the smallest exact fraction, and asserts
    every other tensor bit-exact."""
    path = tmp_path / "q.json"
    c.save(path)
    o = OraclePipeline(g, path)
    fb = _fallback_outputs(g)
    dev = {n: ex.tensors[n].to_host() for n in fb}
    o.run(x, keep=True, overrides=dev)
    worst, exact = 0, 1.0
    for n in fb:
        d = np.abs(dev[n].astype(np.int64) -
                   o.computed[n].reshape(dev[n].shape).astype(np.int64))
        worst, exact = max(worst, int(d.max())), min(exact,
                                                     float((d == 0).mean()))
    checked = 0
    for n, t in ex.tensors.items():
        if n in o.env and n not in fb:
            got = t.to_host()
            np.testing.assert_array_equal(got, o.env[n].reshape(got.shape),
                                          err_msg=n)
            checked += 1
    return worst, exact, checked


def _single_op_graph(kind, shape):
    b = G.GraphBuilder(21, opset=17)
    x = "x"
    if kind == "layernorm":
        c = shape[-1]
        y = b.op("LayerNormalization",
                 [x, b.weight(c, scale=0.5), b.weight(c, scale=0.2)],
                 axis=-1, epsilon=1e-6)
    elif kind == "matmul":  # x @ x^T over the last two axes
        y = b.op("MatMul", [x, b.op("Transpose", [x], perm=[0, 1, 3, 2])])
    elif kind == "matmul_nt":  # B not contiguous along K: a copy is made
        t = b.op("Transpose", [x], perm=[0, 1, 3, 2])
        y = b.op("MatMul", [t, x])
    elif kind == "softmax":
        y = b.op("Softmax", [x], axis=-1)
    else:  # gather of token 0
        y = b.op("Gather", [x, b.const(np.array(0, np.int64))], axis=1)
    y = b.op("Relu", [y])  # an integer layer after the fallback
    return b.build(x, [None] + list(shape[1:]), y)


@pytest.mark.parametrize("quant_type", ["int8", "uint8", "int16"])
@pytest.mark.parametrize("kind,shape", [
    ("layernorm", (3, 17, 64)),
    ("layernorm", (2, 5, 384)),
    ("matmul", (2, 3, 17, 32)),
    ("matmul", (1, 2, 70, 100)),
    ("matmul_nt", (2, 2, 33, 20)),
    ("softmax", (2, 3, 17, 17)),
    ("gather", (3, 9, 48)),
])
def test_fallback_op_within_one_step(hip, tmp_path, quant_type, kind, shape):
    g = _single_op_graph(kind, shape)
    calib = [Stream(30 + i).normal(shape).astype(np.float32) for i in range(2)]
    c = _calibrated(g, quant_type, calib)
    x = Stream(40).normal(shape).astype(np.float32) * np.float32(1.1)
    ex = c.executor({"x": x.shape})
    ex.run({"x": x})
    worst, exact, checked = _check_against_oracle(c, g, tmp_path, x, ex)
    assert worst <= 1, f"{kind}: max difference {worst} steps"
    assert exact >= 0.99, f"{kind}: only {exact:.4f} exact"
    assert checked >= 2


def _tiny_vit():
    return G.vit(seed=5, batch=3, size=32, patch=8, dim=64, depth=2, heads=2,
                 mlp=128, classes=10)


@pytest.mark.parametrize("quant_type", ["int8", "uint8"])
def test_tiny_vit_matches_oracle(hip, tmp_path, quant_type):
    g = _tiny_vit()
    calib = [Stream(50 + i).normal((3, 3, 32, 32)).astype(np.float32)
             for i in range(2)]
    c = _calibrated(g, quant_type, calib)
    x = Stream(60).normal((3, 3, 32, 32)).astype(np.float32)
    # each operator on its own (the scores and probabilities kept)
    ex = c.executor({"images": x.shape}, fuse_attention=False)
    ex.run({"images": x})
    worst, exact, checked = _check_against_oracle(c, g, tmp_path, x, ex)
    assert worst <= 1 and exact >= 0.99, (worst, exact)
    assert checked >= 20


@pytest.mark.parametrize("quant_type", ["int8", "uint8"])
def test_tiny_vit_fused_attention_equals_unfused(hip, quant_type):
    """q k^T -> Softmax -> . v as one launch (int8) gives the three
    launches' results bit for bit: every tensor both passes keep, and the
    logits."""
    g = _tiny_vit()
    calib = [Stream(50 + i).normal((3, 3, 32, 32)).astype(np.float32)
             for i in range(2)]
    c = _calibrated(g, quant_type, calib)
    x = Stream(61).normal((3, 3, 32, 32)).astype(np.float32)
    fused = c.executor({"images": x.shape})
    plain = c.executor({"images": x.shape}, fuse_attention=False)
    n_att = sum(n.startswith("attention:") for n, _ in fused.launches)
    # uint8 activations are stored shifted from their zero points, which
    # the fused kernel does not take: those passes stay unfused
    assert n_att == (2 if quant_type == "int8" else 0), \
        [n for n, _ in fused.launches]
    assert not any(n.startswith("attention:") for n, _ in plain.launches)
    out_f = fused.run({"images": x})
    out_p = plain.run({"images": x})
    common = [n for n in fused.tensors if n in plain.tensors]
    assert len(common) >= 20
    for n in common:
        np.testing.assert_array_equal(fused.tensors[n].to_host(),
                                      plain.tensors[n].to_host(), err_msg=n)
    assert out_f.keys() == out_p.keys()
    for n in out_f:
        np.testing.assert_array_equal(out_f[n], out_p[n], err_msg=n)


def test_tiny_vit_graph_replay_matches_eager(hip):
    g = _tiny_vit()
    calib = [Stream(50).normal((3, 3, 32, 32)).astype(np.float32)]
    c = _calibrated(g, "int8", calib)
    ex = c.executor({"images": (3, 3, 32, 32)})
    x = Stream(62).normal((3, 3, 32, 32)).astype(np.float32)
    eager = ex.run({"images": x})
    for _ in range(3):
        got = ex.run({"images": x}, use_graph=True)
        for k in eager:
            np.testing.assert_array_equal(got[k], eager[k])


def _gemm_block_graph(k, n, act, residual):
    """x [M, k] -> MatMul(+bias) [-> Gelu] [-> + residual (a second
    MatMul of x)]: the weight GEMM forms of a transformer block."""
    b = G.GraphBuilder(31, opset=17)
    w = b.weight(k, n, scale=float(np.sqrt(1.0 / k)))
    y = b.op("MatMul", ["x", w, b.weight(n, scale=0.05)])
    if act:
        y = b.op("Gelu", [y], approximate="tanh")
    if residual:
        r = b.op("MatMul", ["x", b.weight(k, n, scale=float(np.sqrt(1.0 / k))),
                            b.weight(n, scale=0.05)])
        y = b.op("Add", [r, y])
    return b.build("x", [None, k], y)


@pytest.mark.parametrize("quant_type", ["int8", "uint8"])
@pytest.mark.parametrize("m,k,n,act,residual", [
    (1500, 384, 1152, False, False),   # QKV-like, partial row block
    (1100, 256, 384, True, False),     # fc1-like with the Gelu table
    (1030, 1536, 200, False, True),    # fc2-like, residual, partial column block
    (2048, 320, 256, True, True),      # five K steps
    (1024, 128, 256, False, False),    # two K steps: fewer than the stages
])
def test_large_gemm_kernel_bit_exact(hip, tmp_path, quant_type, m, k, n, act,
                                     residual):
    """Weight GEMMs of >= 1024 rows (tile code 0x10400, the library's choice
    of block, 0x10403 / 0x10404, 128 x 128 blocks with 3 / 4 LDS stages
    filled by direct loads, and every other tile code) equal the oracle bit
    for bit."""
    g = _gemm_block_graph(k, n, act, residual)
    calib = [Stream(90 + i).normal((256, k)).astype(np.float32)
             for i in range(2)]
    c = _calibrated(g, quant_type, calib)
    x = Stream(95).normal((m, k)).astype(np.float32)
    path = tmp_path / "q.json"
    c.save(path)
    o = OraclePipeline(g, path)
    o.run(x, keep=True)
    ex = c.executor({"x": x.shape})
    descs = [t for t in ex.tunables]
    assert descs and all({0x10400, 0x10403, 0x10404} <= set(t[2])
                         for t in descs)
    for r in range(max(len(t[2]) for t in descs)):
        for _, d, codes, _ in descs:
            d.tile = codes[r % len(codes)]
        ex.run({"x": x})
        for name, t in ex.tensors.items():
            if name in o.env:
                got = t.to_host()
                np.testing.assert_array_equal(
                    got, o.env[name].reshape(got.shape),
                    err_msg=f"{name}, tiles {[hex(t[1].tile) for t in descs]}")


@pytest.mark.parametrize("rows,cols", [(37, 17), (64, 197), (9, 256),
                                       (12, 300), (5, 512), (64, 1000),
                                       (3, 1024)])
def test_softmax_table_equals_direct(hip, rows, cols):
    """The int8 Softmax through the table of exponentials stores exactly
    what the per-element float64 form stores (same exponentials, same
    summation order), rows of mixed byte ranges included; the forms that
    also write the dequantized graph output agree on it."""
    import torch
    lib = hip.require()
    rng = np.random.default_rng(rows * 1000 + cols)
    x = rng.integers(-128, 128, size=(rows, cols), dtype=np.int64)
    x[0, :] = 17                      # a constant row
    x[1 % rows, :] = rng.integers(-128, -120, size=cols)  # low bytes only
    xd = torch.from_numpy(x.astype(np.int8)).cuda()
    in_scale, in_zp, in_so = 0.0713, 3, 0
    o_scale, o_zp, o_so = 1.0 / 255, -128, 0
    ya = torch.empty_like(xd)
    yb = torch.empty_like(xd)
    tab = torch.empty(65536, dtype=torch.float64, device="cuda")
    s = torch.cuda.current_stream().cuda_stream
    assert lib.qa_d_softmax_table(in_scale, in_zp, in_so, tab.data_ptr(),
                                  s) == 0
    assert lib.qa_d_softmax(xd.data_ptr(), 1, rows, cols, in_scale, in_zp,
                            in_so, ya.data_ptr(), 1, o_scale, o_zp, -128, 127,
                            o_so, s) == 0
    assert lib.qa_d_softmax_lut(xd.data_ptr(), rows, cols, tab.data_ptr(),
                                yb.data_ptr(), o_scale, o_zp, -128, 127,
                                o_so, s) == 0
    torch.cuda.synchronize()
    np.testing.assert_array_equal(yb.cpu().numpy(), ya.cpu().numpy())
    fa = torch.empty((rows, cols), dtype=torch.float32, device="cuda")
    fb = torch.empty_like(fa)
    assert lib.qa_d_softmax_f32(xd.data_ptr(), 1, rows, cols, in_scale,
                                in_zp, in_so, ya.data_ptr(), 1, o_scale, o_zp,
                                -128, 127, o_so, fa.data_ptr(), s) == 0
    assert lib.qa_d_softmax_lut_f32(xd.data_ptr(), rows, cols,
                                    tab.data_ptr(), yb.data_ptr(), o_scale,
                                    o_zp, -128, 127, o_so, fb.data_ptr(),
                                    s) == 0
    torch.cuda.synchronize()
    np.testing.assert_array_equal(yb.cpu().numpy(), ya.cpu().numpy())
    np.testing.assert_array_equal(fb.cpu().numpy(), fa.cpu().numpy())
    want = (ya.cpu().numpy().astype(np.float64) - o_zp) * o_scale
    np.testing.assert_array_equal(fa.cpu().numpy(), want.astype(np.float32))
