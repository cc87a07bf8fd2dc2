"""16-bit convolutions with their weights and activation table in LDS: maps
large enough that a work-group stages the table, channel counts around the
16-channel blocks, one to many K-steps (every depth of the ring), a residual
Add and a Concat copy, inputs past the calibrated range (table clips), all
against the oracle bit for bit."""

import ctypes

import numpy as np
import pytest

from oracle.pipeline import OraclePipeline
from quantanything_amd import graph as G
from quantanything_amd.container import QuantContainer
from quantanything_amd.executor import ConvDesc
from quantanything_amd.synth import Stream

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,cin,cout,k,stride,size,form", [
    (9, 3, 16, 3, 2, 130, "plain"),     # the 4-channel stem
    (4, 3, 24, 5, 1, 66, "plain"),      # 25 taps of it: 7 steps
    (9, 16, 32, 1, 1, 66, "add"),       # one step (of 16 positions)
    (9, 64, 48, 1, 1, 40, "concat"),    # one step
    (4, 128, 64, 1, 1, 48, "add"),      # two steps
    (5, 32, 36, 3, 1, 45, "plain"),     # five steps: rounded up
    (3, 48, 64, 3, 2, 63, "concat"),    # seven
    (2, 64, 20, 3, 1, 61, "add"),       # nine
    (3, 160, 16, 2, 1, 30, "plain"),    # ten
    (1, 256, 64, 3, 1, 9, "add"),       # 36, few tiles
])
def test_bit_exact(hip, tmp_path, n, cin, cout, k, stride, size, form):
    b = G.GraphBuilder(61)
    y = b.silu(b.conv("x", cin, cout, k, stride, w_scale=(cin * k * k) ** -.5))
    if form != "plain":
        r = b.op("Relu", [b.conv("x", cin, cout, k, stride,
                                 w_scale=(cin * k * k) ** -.5)])
        if form == "add":
            y = b.op("Add", [r, y])
        else:
            y = b.op("Concat", [r, y], axis=1)
    g = b.build("x", [None, cin, size, size], y)
    shape = (n, cin, size, size)
    q = QuantContainer(g, "int16", per_channel=True)
    q.calibrate([Stream(12).normal((1,) + shape[1:]).astype(np.float32)])
    q.save(tmp_path / "q.json")
    data = Stream(13).normal(shape, 1.4).astype(np.float32)
    oracle = OraclePipeline(g, str(tmp_path / "q.json"))
    oracle.run(data, keep=True)
    ex = q.executor({"x": shape})
    ds = [d for d in ex.keep if isinstance(d, ConvDesc)]
    assert all(d.wsplit for d in ds) and any(d.epi_plan for d in ds)
    # every channel block: the library's choice, then 1, 2 and 4
    for code in (0, 0x11011, 0x11012, 0x11014):
        for d in ds:
            d.tile = code
        ex.run({"x": data})
        checked = 0
        for name, t in ex.tensors.items():
            if name in oracle.env:
                got = t.to_host()
                np.testing.assert_array_equal(
                    got, oracle.env[name].reshape(got.shape),
                    err_msg=f"{name} {code:#x}")
                checked += 1
        assert checked >= 1


@pytest.mark.parametrize("other", ["shorter", "int8", "off 16"])
def test_other_plans_are_ignored(hip, other):
    """A descriptor whose epi_plan is not the plan of its own table (of a
    shorter table, an int8 epilogue's, off its alignment) reads the table
    itself."""
    import torch

    b = G.GraphBuilder(62)
    y = b.silu(b.conv("x", 16, 32, 1, 1, w_scale=0.25))
    shape = (9, 16, 66, 66)
    g = b.build("x", [None, *shape[1:]], y)
    q = QuantContainer(g, "int16", per_channel=True)
    q.calibrate([Stream(12).normal((1,) + shape[1:]).astype(np.float32)])
    data = Stream(13).normal(shape, 1.4).astype(np.float32)
    ex = q.executor({"x": shape})
    want = ex.run({"x": data})[g.outputs[0]].copy()
    d, = [d for d in ex.keep if isinstance(d, ConvDesc)]
    lib, n = hip.library(), int(d.lut_len)
    assert d.epi_plan and n > 40
    lut = np.arange(40 if other == "shorter" else n, dtype=np.int32)
    plan = np.zeros(lib.qa_lut_i16_plan_bytes(len(lut)), np.uint8)
    assert lib.qa_plan_lut_i16(lut.ctypes.data, len(lut),
                               plan.ctypes.data) == 1
    if other == "int8":  # its header: clip bounds, shift, flags
        plan = np.zeros(64, np.uint8)
        plan[:16].view(np.int32)[:] = (-128, 127, 1 << 16, 0)
    dev = torch.from_numpy(np.concatenate(
        [np.zeros(8 if other == "off 16" else 0, np.uint8), plan])).cuda()
    d.epi_plan = dev.data_ptr() + (8 if other == "off 16" else 0)
    np.testing.assert_array_equal(ex.run({"x": data})[g.outputs[0]], want)


@pytest.mark.parametrize("n,cin,cout,k,size,form", [
    (3, 16, 18, 3, 13, "plain"), (2, 32, 34, 1, 12, "add"),
    (2, 48, 22, 3, 11, "concat"), (3, 3, 18, 3, 15, "add"),
    (2, 4, 10, 3, 14, "concat"),  # pixels of 4 channels
    (1, 576, 20, 3, 7, "plain"), (1, 560, 32, 3, 6, "add")])
def test_form_without_lds(hip, tmp_path, n, cin, cout, k, size, form):
    """The byte split without its weights in LDS, where that form does not
    apply (pixels off 4 channels, weights past the LDS): every tile code,
    plain, with a residual Add and with a Concat copy."""
    b = G.GraphBuilder(63)
    x = b.op("Relu", [b.conv("x", 5, cin, 1)]) if cin > 4 else "x"
    if form == "add":
        r = b.op("Relu", [b.conv(x, cin, cout, 1)])
    y = b.silu(b.conv(x, cin, cout, k, w_scale=(cin * k * k) ** -.5))
    if form == "add":
        y = b.op("Add", [r, y])
    elif form == "concat":
        y = b.op("Concat", [b.op("MaxPool", [y], kernel_shape=[1, 1],
                                 strides=[1, 1]), y], axis=1)
    shape = (n, 5 if cin > 4 else cin, size, size)
    g = b.build("x", [None, *shape[1:]], y)
    q = QuantContainer(g, "int16", per_channel=True)
    q.calibrate([Stream(14).normal(shape).astype(np.float32)])
    q.save(tmp_path / "q.json")
    data = Stream(15).normal(shape, 1.3).astype(np.float32)
    oracle = OraclePipeline(g, str(tmp_path / "q.json"))
    oracle.run(data, keep=True)
    ex = q.executor({"x": shape})
    ds = [d for d in ex.keep if isinstance(d, ConvDesc) and d.wsplit and
          d.KH == k and not
          hip.library().qa_conv_split_lds(ctypes.byref(d))]
    assert ds and all((d.res if form == "add" else d.y2 if form == "concat"
                       else True) for d in ds[-1:])
    for code in [0] + [0x11000 | wm | tm << 4 for tm in (1, 2)
                       for wm in (1, 2, 4)]:
        for d in ds:
            d.tile = code
        ex.run({"x": data})
        checked = 0
        for name, t in ex.tensors.items():
            if name in oracle.env:
                got = t.to_host()
                np.testing.assert_array_equal(
                    got, oracle.env[name].reshape(got.shape),
                    err_msg=f"{name} {code:#x}")
                checked += 1
        assert checked >= 1
