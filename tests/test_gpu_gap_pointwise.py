"""GlobalAveragePool over 16-byte rows (qa_d_gap: whole and partial channel
chunks, few and many pixels, extremes of int8 and int16) against NumPy and
Python integers, and pointwise convolutions run as GEMMs over their pixels
(the narrow kernel below 1024 of its blocks, the large-GEMM blocks past that
or with a residual: partial row and column blocks, a Concat copy) against the
oracle, every value equal."""

import numpy as np
import pytest

from oracle.pipeline import OraclePipeline
from quantanything_amd import graph as G
from quantanything_amd.container import QuantContainer
from quantanything_amd.synth import Stream
from quantanything_amd.utils import multiply_by_quantized_multiplier

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("code", [1, 2])
@pytest.mark.parametrize("n,c,hw,fill", [
    (3, 64, 49, None), (2, 20, 1, None), (1, 300, 511, None),
    (2, 7, 512, None), (5, 128, 3136, None), (2, 72, 2000, -1),
    (2, 65, 700, 1)])
def test_gap_rows(hip, code, n, c, hw, fill):
    import torch

    t = np.int8 if code == 1 else np.int16
    info = np.iinfo(t)
    rng = np.random.default_rng(c)
    sp = -(-c // 16) * 16
    x = rng.integers(info.min, info.max + 1, (n, hw, sp)).astype(t)
    if fill is not None:
        x[:] = info.min if fill < 0 else info.max
    zi, so, m, s, zo = 3, 1, 1400000000, 6, -2
    xd = torch.from_numpy(x).cuda()
    y = torch.full((n, c + 3), 9, dtype=xd.dtype, device="cuda")
    assert hip.library().qa_d_gap(
        xd.data_ptr(), code, hw * sp, 1, sp, n, c, hw, zi, so, m, s, zo,
        int(info.min), int(info.max), y.data_ptr(), code, c + 3, 0,
        None) == 0
    acc = x[:, :, :c].astype(np.int64).sum(1) + hw * (so - zi)
    want = np.clip(multiply_by_quantized_multiplier(acc, m, s) + zo,
                   info.min, info.max)
    got = y.cpu().numpy()
    np.testing.assert_array_equal(got[:, :c], want.astype(t))
    assert (got[:, c:] == 9).all()


@pytest.mark.parametrize("n,c,hw,sp,off", [
    (3, 20, 49, 20, 0), (2, 64, 700, 68, 4), (1, 300, 3, 320, 12),
    (2, 12, 3136, 24, 12), (2, 4, 1, 4, 0), (300, 256, 130, 256, 0),
    (3, 128, 128, 128, 0), (3, 128, 129, 128, 0), (3, 20, 511, 32, 0),
    (3, 20, 512, 32, 0), (70, 300, 513, 304, 0),  # words of 4 channels
    (3, 18, 24, 32, 0), (3, 18, 25, 32, 0),
    (2, 18, 49, 20, 0), (2, 20, 49, 21, 1), (2, 18, 8, 32, 0),
    (700, 130, 16, 144, 0)])  # a channel a thread
def test_gap_words_and_channels(hip, n, c, hw, sp, off):
    """Rows on 4 bytes alone (a Split half, a caller's dense rows) and on
    none, few pixels and many images."""
    import torch

    rng = np.random.default_rng(c + hw)
    x = rng.integers(-128, 128, (n, hw, sp)).astype(np.int8)
    x = np.concatenate([x.reshape(-1), np.zeros(64, np.int8)])
    zi, so, m, s, zo = 3, 1, 1400000000, 6, -2
    xd = torch.from_numpy(x).cuda()
    y = torch.full((n, c + 3), 9, dtype=torch.int8, device="cuda")
    assert hip.library().qa_d_gap(
        xd.data_ptr() + off, 1, hw * sp, 1, sp, n, c, hw, zi, so, m, s, zo,
        -128, 127, y.data_ptr(), 1, c + 3, 0, None) == 0
    rows = np.stack([x[off + i * hw * sp:][:hw * sp].reshape(hw, sp)[:, :c]
                     for i in range(n)])
    acc = rows.astype(np.int64).sum(1) + hw * (so - zi)
    want = np.clip(multiply_by_quantized_multiplier(acc, m, s) + zo, -128,
                   127)
    got = y.cpu().numpy()
    np.testing.assert_array_equal(got[:, :c], want.astype(np.int8))
    assert (got[:, c:] == 9).all()


@pytest.mark.parametrize("qt", ["int8", "uint8"])
@pytest.mark.parametrize("cin,cout,size,form", [
    (64, 128, 19, "plain"), (128, 132, 16, "add"), (64, 200, 18, "concat"),
    (192, 130, 17, "plain"),
    (64, 128, 46, "plain"), (64, 200, 47, "concat"), (192, 130, 38, "plain")])
def test_pointwise_as_gemm(hip, tmp_path, qt, cin, cout, size, form):
    b = G.GraphBuilder(43)
    x = b.op("Relu", [b.conv("x", 4, cin, 1)])
    y = b.silu(b.conv(x, cin, cout, 1))
    if form == "add":
        y = b.op("Add", [b.op("Relu", [b.conv("x", 4, cout, 1)]), y])
    elif form == "concat":
        y = b.op("Concat", [b.op("MaxPool", [y], kernel_shape=[1, 1],
                                 strides=[1, 1]), y], axis=1)
    g = b.build("x", [None, 4, size, size], y)
    shape = (4, 4, size, size)
    q = QuantContainer(g, qt, per_channel=True)
    q.calibrate([Stream(7).normal(shape).astype(np.float32)])
    q.save(tmp_path / "q.json")
    data = Stream(8).normal(shape, 1.2).astype(np.float32)
    oracle = OraclePipeline(g, str(tmp_path / "q.json"))
    oracle.run(data, keep=True)
    ex = q.executor({"x": shape})
    ex.run({"x": data})
    checked = 0
    for name, t in ex.tensors.items():
        if name in oracle.env:
            got = t.to_host()
            np.testing.assert_array_equal(
                got, oracle.env[name].reshape(got.shape), err_msg=name)
            checked += 1
    assert checked >= 2
