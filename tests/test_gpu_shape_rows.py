"""The 16-byte forms of MaxPool, Pad and the int8 rescale against NumPy on
the same stored values, every value equal: channel counts around the 16-byte
chunks, windows inside and across the border, dilations, a padding value
above every tap, pools of whole images, Pads of every axis order."""

import ctypes

import numpy as np
import pytest

from quantanything_amd.executor import MaxPoolDesc, NdCopy, PadDesc
from quantanything_amd.utils import multiply_by_quantized_multiplier

pytestmark = pytest.mark.gpu
TYPES = {1: np.int8, 2: np.int16}


def _dev(a):
    import torch

    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("code", [1, 2])
@pytest.mark.parametrize("n,c,h,w,k,s,dl,pad", [
    (2, 32, 17, 19, (5, 5), (1, 1), (1, 1), (2, 2)),
    (3, 20, 12, 9, (3, 3), (2, 2), (1, 1), (1, 1)),
    (2, 7, 8, 8, (2, 2), (2, 2), (1, 1), (0, 0)),
    (2, 48, 15, 14, (3, 3), (1, 2), (2, 1), (2, 1)),
    (1, 24, 9, 11, (3, 5), (1, 1), (1, 1), (1, 2)),
    (3, 40, 23, 21, (23, 21), (1, 1), (1, 1), (0, 0)),  # the whole image
    (2, 16, 20, 20, (9, 9), (3, 3), (1, 1), (4, 4)),
    (1, 300, 9, 8, (9, 8), (1, 1), (1, 1), (0, 0)),
    (5, 72, 7, 7, (7, 7), (1, 1), (1, 1), (0, 0)),  # a work-group an output
    (2, 24, 11, 12, (4, 4), (2, 2), (1, 1), (1, 1)),
    (3, 33, 8, 9, (2, 8), (1, 1), (2, 1), (0, 2)),
    (9, 256, 17, 16, (4, 5), (1, 1), (1, 1), (2, 2)),  # 41472, 82944 chunks
    (2, 16, 9, 9, (5, 3), (2, 2), (1, 1), (1, 1)),
    # partial last chunks past the size from which they take chunks
    (5, 100, 25, 24, (5, 5), (1, 1), (1, 1), (2, 2)),
    (4, 33, 56, 57, (3, 3), (1, 1), (1, 1), (1, 1)),
    (3, 24, 151, 150, (2, 2), (2, 2), (1, 1), (0, 0)),
    (1, 36, 110, 111, (3, 2), (1, 1), (1, 1), (0, 1))])
@pytest.mark.parametrize("high", [False, True])
def test_maxpool_chunks(hip, code, n, c, h, w, k, s, dl, pad, high):
    t = TYPES[code]
    rng = np.random.default_rng(n * c + h)
    cs = -(-c // 16) * 16
    info = np.iinfo(t)
    x = rng.integers(info.min, info.max + 1, (n, h, w, cs)).astype(t)
    pv = info.max if high else info.min
    oh = (h + 2 * pad[0] - dl[0] * (k[0] - 1) - 1) // s[0] + 1
    ow = (w + 2 * pad[1] - dl[1] * (k[1] - 1) - 1) // s[1] + 1
    big = np.full((n, h + 2 * pad[0], w + 2 * pad[1], c), pv, t)
    big[:, pad[0]:pad[0] + h, pad[1]:pad[1] + w] = x[..., :c]
    want = np.full((n, oh, ow, c), info.min, t)
    for ky in range(k[0]):
        for kx in range(k[1]):
            y0, x0 = ky * dl[0], kx * dl[1]
            want = np.maximum(want, big[:, y0:y0 + (oh - 1) * s[0] + 1:s[0],
                                        x0:x0 + (ow - 1) * s[1] + 1:s[1]])
    xd, yd = _dev(x), _dev(np.full((n, oh, ow, cs), 55, t))
    d = MaxPoolDesc()
    d.x, d.code, d.y = xd.data_ptr(), code, yd.data_ptr()
    d.x_sn, d.x_sc, d.x_sh, d.x_sw = h * w * cs, 1, w * cs, cs
    d.y_sn, d.y_sc, d.y_sh, d.y_sw = oh * ow * cs, 1, ow * cs, cs
    d.N, d.C, d.H, d.W, d.OH, d.OW = n, c, h, w, oh, ow
    (d.KH, d.KW), (d.SH, d.SW), (d.DH, d.DW) = k, s, dl
    (d.PT, d.PL), d.pad = pad, int(pv)
    assert hip.library().qa_d_maxpool(ctypes.byref(d), None) == 0
    got = yd.cpu().numpy()
    np.testing.assert_array_equal(got[..., :c], want)
    assert (got[..., c:] == 55).all()


@pytest.mark.parametrize("code", [1, 2])
@pytest.mark.parametrize("shape,lo,hi,order", [
    ((2, 64, 9, 7), (0, 2, 1, 2), (0, 1, 2, 1), (0, 2, 3, 1)),
    ((3, 20, 4, 5), (1, 0, 0, 3), (0, 5, 2, 0), (0, 2, 3, 1)),
    ((2, 5, 6, 40), (0, 1, 1, 7), (1, 0, 1, 9), (0, 1, 2, 3)),
    ((4, 33), (2, 3), (1, 2), (0, 1)), ((33, 18), (0, 4), (1, 1), (1, 0)),
    ((2, 3, 4, 17), (0, 0, 0, 16), (0, 0, 0, 1), (3, 1, 0, 2)),
    # past the size from which a thread takes 16 bytes of a row
    ((4, 70, 33, 31), (0, 2, 1, 2), (0, 1, 2, 1), (0, 2, 3, 1)),
    ((1500, 533), (2, 3), (1, 2), (0, 1)),
    ((533, 1500), (0, 4), (1, 1), (1, 0))])
def test_pad_rows(hip, code, shape, lo, hi, order):
    t = TYPES[code]
    rng = np.random.default_rng(sum(shape))
    nd = len(shape)
    x = rng.integers(-100, 100, shape).astype(t)
    want = np.pad(x, list(zip(lo, hi)), constant_values=-77)
    # both tensors laid out with axis order[-1] innermost
    xm = np.ascontiguousarray(x.transpose(order))
    ym = np.zeros([want.shape[a] for a in order], t)
    xd, yd = _dev(xm), _dev(np.concatenate([ym.reshape(-1),
                                            np.full(40, 9, t)]))
    d = PadDesc()
    d.x, d.code, d.y, d.ndim = xd.data_ptr(), code, yd.data_ptr(), nd
    for pos, a in enumerate(order):
        d.shape[a], d.lo[a], d.xshape[a] = want.shape[a], lo[a], shape[a]
        d.xs[a] = int(np.prod(xm.shape[pos + 1:], dtype=np.int64))
        d.ys[a] = int(np.prod(ym.shape[pos + 1:], dtype=np.int64))
    d.fill = -77
    assert hip.library().qa_d_pad_nd(ctypes.byref(d), None) == 0
    got = yd.cpu().numpy()
    np.testing.assert_array_equal(
        got[:ym.size].reshape(ym.shape), want.transpose(order))
    assert (got[ym.size:] == 9).all()


@pytest.mark.parametrize("code", [1, 2])
@pytest.mark.parametrize("shape,xst,yst,off", [
    ((3, 17, 4, 5), (640, 1, 160, 32), (480, 1, 120, 24), 5),
    ((9, 31, 40, 41), (104960, 1, 2624, 64), (82000, 1, 2050, 50), 31),
    ((2, 24, 90, 91), (0, 1, 4368, 48), (262080, 1, 2912, 32), 24),
    ((1700, 501), (512, 1), (503, 1), 1), ((30, 37), (37, 1), (64, 1), 0),
    ((501, 1700), (1, 512), (1, 503), 3), ((40, 9000), (9001, 1), (9000, 1), 0),
    # the output's rows not contiguous, or its other axis at stride 1
    ((900, 900), (900, 1), (1801, 2), 0), ((900, 1), (16, 1), (1, 1), 0)])
def test_copy_rows(hip, code, shape, xst, yst, off):
    """Plain copies of views off the 16-byte grid (a Split's half, a batch
    read again from one image, odd matrices), on each side of the size from
    which a thread takes 16 bytes of a row."""
    import torch

    t = TYPES[code]
    info = np.iinfo(t)
    rng = np.random.default_rng(sum(shape))
    size = off + 1 + sum((n - 1) * s for n, s in zip(shape, xst))
    x = rng.integers(info.min, info.max + 1, size).astype(t)
    ysize = 1 + sum((n - 1) * s for n, s in zip(shape, yst))
    xd, yd = _dev(x), _dev(np.full(ysize + 40, 55, t))
    d = NdCopy()
    d.x, d.x_code = xd.data_ptr() + off * code, code
    d.y, d.y_code, d.ndim = yd.data_ptr(), code, len(shape)
    for k, v in enumerate(zip(shape, xst, yst)):
        d.shape[k], d.xs[k], d.ys[k] = v
    d.qmin, d.qmax = -(1 << 62), 1 << 62
    assert hip.library().qa_d_copy_nd(ctypes.byref(d), None) == 0
    want = torch.full((ysize + 40,), 55, dtype=yd.dtype)
    torch.as_strided(want, shape, yst).copy_(
        torch.as_strided(torch.from_numpy(x), shape, xst, off))
    np.testing.assert_array_equal(yd.cpu().numpy(), want.numpy())


@pytest.mark.parametrize("rows,cols,xs,ys,m,s,qmin,qmax", [
    (1000, 32, 32, 128, (1 << 30) + 12345, 0, -128, 127),
    (77, 40, 64, 48, 1500000000, -1, -100, 90),
    (5, 16, 16, 16, 1 << 30, -1, -128, 127),
    (3, 1000, 1008, 1024, 2000000001, 3, -128, 127),
    (4096, 17, 32, 32, -1100000000, 1, -128, 127),
    # a partial last chunk past the size from which chunks pay
    (16384, 17, 32, 48, -1100000000, 1, -128, 127),
    (9000, 30, 32, 32, 1500000000, -1, -100, 90)])
def test_rescale_rows(hip, rows, cols, xs, ys, m, s, qmin, qmax):
    rng = np.random.default_rng(cols)
    x = rng.integers(-128, 128, (rows, xs)).astype(np.int8)
    xd, yd = _dev(x), _dev(np.full((rows, ys), 3, np.int8))
    zi, zo, si, so = 5, -3, 0, 0
    assert hip.library().qa_d_rescale(
        xd.data_ptr(), 1, xs, yd.data_ptr(), 1, ys, rows, cols, zi, m, s, zo,
        qmin, qmax, si, so, None) == 0
    v = x[:, :cols].astype(np.int64) + si - zi
    want = np.clip(multiply_by_quantized_multiplier(v, m, s) + zo, qmin,
                   qmax) - so
    got = yd.cpu().numpy()
    np.testing.assert_array_equal(got[:, :cols], want.astype(np.int8))
    assert (got[:, cols:] == 3).all()
