"""Depthwise int8 convolutions on the matrix cores (weights packed in layout
2) against the oracle, every tensor bit for bit: channel counts around the
16-channel blocks, kernels on each side of the 4, 12, 28 and 52 tap steps,
strides, dilations and paddings on odd sizes, a residual Add, a Concat copy,
uint8 weights whose offset needs the window sums. Kernels of more than 52
taps keep the general path."""

import numpy as np
import pytest

from oracle.pipeline import OraclePipeline
from quantanything_amd import graph as G
from quantanything_amd.container import QuantContainer
from quantanything_amd.executor import ConvDesc
from quantanything_amd.synth import Stream

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("qt", ["int8", "uint8"])
@pytest.mark.parametrize("c,k,stride,pad,dil,size,form", [
    (8, 1, 1, 0, 1, 5, "plain"), (16, 2, 2, 0, 1, 9, "plain"),
    (24, 3, 1, 1, 1, 17, "plain"), (128, 3, 2, 1, 1, 14, "plain"),
    (20, 3, 1, 2, 2, 11, "add"), (40, 3, 1, 1, 1, 13, "concat"),
    (33, 5, 1, 2, 1, 12, "add"), (64, 5, 2, 2, 1, 19, "concat"),
    (16, 7, 1, 3, 1, 10, "plain"), (9, 8, 1, 4, 1, 9, "plain")])
def test_depthwise_bit_exact(hip, tmp_path, qt, c, k, stride, pad, dil, size,
                             form):
    b = G.GraphBuilder(41)
    x = b.op("Relu", [b.conv("x", 4, c, 1)])
    y = b.silu(b.conv(x, c, c, k, stride, pad=pad, dilation=dil, groups=c))
    if form == "add":
        y = b.op("Add", [x, y])
    elif form == "concat":
        y = b.op("Concat", [b.op("MaxPool", [y], kernel_shape=[1, 1],
                                 strides=[1, 1]), y], axis=1)
    g = b.build("x", [None, 4, size, size], y)
    shape = (3, 4, size, size)
    q = QuantContainer(g, qt, per_channel=True)
    q.calibrate([Stream(5).normal(shape).astype(np.float32)])
    q.save(tmp_path / "q.json")
    data = Stream(6).normal(shape, 1.2).astype(np.float32)
    oracle = OraclePipeline(g, str(tmp_path / "q.json"))
    oracle.run(data, keep=True)
    ex = q.executor({"x": shape})
    ex.run({"x": data})
    layouts = [(d.w_code, d.w_layout) for d in ex.keep
               if isinstance(d, ConvDesc) and d.G > 1]
    assert layouts == [(1, 2) if k * k <= 52 else (4, 0)]
    checked = 0
    for name, t in ex.tensors.items():
        if name in oracle.env:
            got = t.to_host()
            np.testing.assert_array_equal(
                got, oracle.env[name].reshape(got.shape), err_msg=name)
            checked += 1
    assert checked >= 2
