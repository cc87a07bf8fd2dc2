"""Float NCHW <-> quantized channels-last (qa_d_quantize_nhwc for more than 4
channels or 16-bit storage, qa_d_dequantize_nchw) against NumPy: float64
quotients rounded half to even, products in float64, every value equal.
Sizes around the 16-byte channel chunks and the 4-pixel groups, strided and
misaligned pixels, near-ties, infinities and NaN."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CODES = {1: (np.int8, 128, 0, 255), 2: (np.int16, 32768, 0, 65535)}


@pytest.mark.parametrize("code,n,c,hw,sp,shift", [
    (1, 1, 5, 1, 16, 0), (1, 2, 24, 57 * 57, 32, 0), (1, 3, 16, 12, 16, 0),
    (1, 8, 64, 56 * 56, 64, 0),
    (1, 2, 7, 9, 7, 0), (1, 2, 20, 10, 21, 1),  # element stores
    (2, 3, 3, 224 * 224, 4, 0), (2, 2, 9, 25, 9, 0),
    (2, 6, 3, 224 * 224, 4, 0), (2, 340, 1, 784, 4, 0),  # four pixels
    (2, 5, 1, 784, 4, 0), (2, 2, 2, 9, 4, 0), (2, 2, 24, 49, 24, 0),
    (2, 1, 8, 64, 8, 1), (2, 64, 40, 36, 40, 0)])
def test_planes_round_trip(hip, code, n, c, hw, sp, shift):
    import torch

    lib = hip.library()
    dt, so, qmin, qmax = CODES[code]
    scale, zp = 0.037, 130
    rng = np.random.default_rng(code * 1000 + c)
    x = rng.normal(0, 60 * scale, (n, c, hw)).astype(np.float32)
    flat = x.reshape(-1)
    k = flat.size // 2  # ties and near-ties of the rounding
    ties = ((rng.integers(-100, 100, k) + 0.5) * scale).astype(np.float32)
    flat[:k] = ties
    flat[k:k + 4][:flat.size - k] = [np.inf, -np.inf, np.nan, 1e30][
        :flat[k:k + 4].size]
    s = torch.cuda.current_stream().cuda_stream
    xd = torch.from_numpy(x).cuda()
    buf = torch.full((n * hw * sp + 64,), 77, dtype=torch.int8 if code == 1
                     else torch.int16, device="cuda")
    y = buf[shift:]
    assert lib.qa_d_quantize_nhwc(xd.data_ptr(), n, c, hw, y.data_ptr(), code,
                                  sp, scale, zp, qmin, qmax, so, s) == 0
    with np.errstate(invalid="ignore"):
        v = np.rint(x.astype(np.float64) / scale) + zp
        q = np.where(np.isnan(v), -2.0**31, np.clip(v, qmin, qmax))
    want = (q.astype(np.int64) - so).astype(dt)
    got = y[:n * hw * sp].cpu().numpy().reshape(n, hw, sp)
    np.testing.assert_array_equal(got[:, :, :c], want.transpose(0, 2, 1))
    assert not got[:, :, c:].any()
    assert (buf.cpu().numpy()[shift + n * hw * sp:] == 77).all()
    # the way back, from a channel offset too (a Split view)
    for c0 in {0, c // 2}:
        yf = torch.full((n * (c - c0) * hw + 8,), 5.0, device="cuda")
        assert lib.qa_d_dequantize_nchw(
            y[c0:].data_ptr(), code, hw * sp, sp, n, c - c0, hw,
            yf.data_ptr(), scale, zp, so, s) == 0
        back = ((got[:, :, c0:c].astype(np.int64) + so - zp) * scale).astype(
            np.float32).transpose(0, 2, 1)
        out = yf.cpu().numpy()
        np.testing.assert_array_equal(out[:n * (c - c0) * hw],
                                      back.reshape(-1))
        assert (out[n * (c - c0) * hw:] == 5.0).all()


@pytest.mark.parametrize("code,c,hw,sp", [
    (1, 40, 36, 48), (1, 7, 9, 7),     # tiles; any pixel stride
    (2, 40, 36, 40), (2, 3, 20, 4),    # tiles; one pixel a thread
    (2, 3, 1 << 17, 4)])               # four
@pytest.mark.parametrize("scale", [2.0**-60, 1e-12, 0.037, 2.0**60])
def test_values_past_float32_quotients(hip, code, c, hw, sp, scale):
    """Finite values whose quotient by the scale passes float32 saturate on
    their own side."""
    import torch

    dt, so, qmin, qmax = CODES[code]
    zp = 130
    top = np.finfo(np.float32).max
    ext = np.array([top, 3.4e38, 1e38, 1.3e37, 1e37, 1e30, 1e20, 0.0,
                    np.inf], np.float32)
    x = np.resize(np.concatenate([ext, -ext, [np.nan]]),
                  (2, c, hw)).astype(np.float32)
    xd = torch.from_numpy(x).cuda()
    y = torch.full((2 * hw * sp,), 77, dtype=torch.int8 if code == 1
                   else torch.int16, device="cuda")
    assert hip.library().qa_d_quantize_nhwc(
        xd.data_ptr(), 2, c, hw, y.data_ptr(), code, sp, scale, zp, qmin,
        qmax, so, torch.cuda.current_stream().cuda_stream) == 0
    with np.errstate(invalid="ignore"):
        v = np.rint(x.astype(np.float64) / scale) + zp
        q = np.where(np.isnan(v), -2.0**31, np.clip(v, qmin, qmax))
    want = (q.astype(np.int64) - so).astype(dt)
    got = y.cpu().numpy().reshape(2, hw, sp)
    np.testing.assert_array_equal(got[:, :, :c], want.transpose(0, 2, 1))


@pytest.mark.parametrize("qt", ["int8", "int16"])
def test_output_of_many_channels(hip, qt):
    """More channels than the one-launch dequantization's grid takes: a
    dense copy first."""
    from quantanything_amd import graph as G
    from quantanything_amd.container import QuantContainer
    from quantanything_amd.synth import Stream

    shape = (1, 65535 * 16 + 16, 2, 1)
    b = G.GraphBuilder(3)
    g = b.build("x", [None, *shape[1:]],
                b.op("MaxPool", ["x"], kernel_shape=[1, 1], strides=[1, 1]))
    data = Stream(4).normal(shape).astype(np.float32)
    q = QuantContainer(g, qt, per_channel=True)
    q.calibrate([data])
    ex = q.executor({"x": shape})
    out = ex.run({"x": data})[g.outputs[0]]
    t = ex.tensors[g.outputs[0]]
    v = np.clip(np.rint(data.astype(np.float64) / t.qp.scale) + t.qp.zp,
                t.qp.qmin, t.qp.qmax)
    np.testing.assert_array_equal(
        out, ((v - t.qp.zp) * t.qp.scale).astype(np.float32))
