"""Gemms and convolutions whose operands sit off the 16-byte grid (odd
feature counts, odd channel halves, rows of a padded input, chains of odd
Gemms) on the int8 matrix cores, against the oracle bit for bit; offsets of
uint8 weights read the padding."""

import numpy as np
import pytest

from oracle.pipeline import OraclePipeline
from quantanything_amd import graph as G
from quantanything_amd.container import QuantContainer
from quantanything_amd.executor import ConvDesc
from quantanything_amd.synth import Stream

pytestmark = pytest.mark.gpu


def _check(g, qt, shape, tmp_path, rows=None):
    name = g.input_names[0]
    q = QuantContainer(g, qt, per_channel=True)
    q.calibrate([Stream(9).normal((rows or shape[0],) + shape[1:])
                 .astype(np.float32)])
    q.save(tmp_path / "q.json")
    data = Stream(10).normal(shape, 1.2).astype(np.float32)
    oracle = OraclePipeline(g, str(tmp_path / "q.json"))
    oracle.run(data, keep=True)
    ex = q.executor({name: shape})
    out = ex.run({name: data})
    ints = ex.integer_outputs()
    for n in g.outputs:
        np.testing.assert_array_equal(
            ints[n], oracle.env[n].reshape(ints[n].shape))
        assert out[n].shape == ints[n].shape
    checked = 0
    for n, t in ex.tensors.items():
        if n in oracle.env:
            got = t.to_host()
            np.testing.assert_array_equal(
                got, oracle.env[n].reshape(got.shape), err_msg=n)
            checked += 1
    assert checked >= 2
    return [d.w_code for d in ex.keep if isinstance(d, ConvDesc)]


@pytest.mark.parametrize("qt", ["int8", "uint8"])
@pytest.mark.parametrize("m,sizes", [
    (1, [17, 5]), (65, [100, 77]), (33, [63, 65, 31]), (1100, [129, 140, 9]),
    (7, [48, 64, 33]), (130, [1, 200]),
    (9, [80, 48, 208, 17]), (300, [1040, 16])])  # rows of whole chunks, dense
def test_odd_gemms(hip, tmp_path, qt, m, sizes):
    b = G.GraphBuilder(51)
    y = "x"
    for k, n in zip(sizes, sizes[1:]):
        y = b.op("Gemm", [y, b.weight(k, n, scale=k ** -0.5),
                          b.weight(n, scale=0.1)])
        if n != sizes[-1]:
            y = b.silu(y)
    codes = _check(b.build("x", [None, sizes[0]], y), qt, (m, sizes[0]),
                   tmp_path, rows=64)
    assert set(codes) == {1}


@pytest.mark.parametrize("qt", ["int8", "uint8"])
@pytest.mark.parametrize("c,k,size", [(24, 3, 9), (11, 3, 12), (31, 1, 8)])
def test_odd_channel_halves(hip, tmp_path, qt, c, k, size):
    """Convolutions of Split halves that start off the 16-byte grid."""
    b = G.GraphBuilder(52)
    y = b.silu(b.conv("x", 5, 2 * c, 1))
    a, d = b.op("Split", [y, b.const(np.array([c, c], np.int64))], n_out=2,
                axis=1)
    d = b.op("Add", [d, b.silu(b.conv(d, c, c, k))])
    y = b.silu(b.conv(b.op("Concat", [a, d], axis=1), 2 * c, 16, 1))
    y = b.op("Flatten", [b.op("GlobalAveragePool", [y])], axis=1)
    codes = _check(b.build("x", [None, 5, size, size], y), qt,
                   (2, 5, size, size), tmp_path)
    assert set(codes) == {1}


def test_other_readers_see_the_rows(hip, tmp_path):
    """A Gemm's odd output read by a Gemm and a Concat stays dense."""
    b = G.GraphBuilder(53)
    h = b.op("Gemm", ["x", b.weight(30, 37, scale=0.2),
                      b.weight(37, scale=0.1)])
    z = b.op("Gemm", [h, b.weight(37, 21, scale=0.2),
                      b.weight(21, scale=0.1)])
    y = b.op("Concat", [h, z], axis=1)
    _check(b.build("x", [None, 30], [y, z]), "int8", (19, 30), tmp_path,
           rows=64)


@pytest.mark.parametrize("m,k,n", [
    (1, 16, 1), (19, 48, 5), (130, 80, 17), (300, 208, 33), (77, 592, 65),
    (260, 1040, 131), (1030, 144, 250), (64, 1264, 37), (515, 2064, 258)])
def test_gemm_rows_off_the_grid(hip, m, k, n):
    """Every kernel a GEMM descriptor can take, K a multiple of 16 alone and
    output rows of any width, against 64-bit integers; the bytes after the
    output stay."""
    import torch

    from quantanything_amd.executor import DeviceExecutor
    from quantanything_amd.workloads import GemmWorkload

    w = GemmWorkload(seed=m + n, M=m, K=k, N=n)
    w.y = torch.full((m * n + 64,), 77, dtype=torch.int8, device="cuda")
    w.d.y = w.y.data_ptr()
    g = w.spec
    acc = (g["a"].astype(np.int64) - g["zp_in"]) @ g["w"].astype(np.int64)
    t = 31 + g["shift"]
    q = ((acc + g["bias"]) * g["mult"] + (1 << (t - 1))) >> t
    want = (np.clip(q + g["zp_out"], g["qmin"], g["qmax"]) - 128)
    codes = DeviceExecutor.tile_candidates(w.d)
    assert any(c >> 13 & 1 for c in codes) == (k <= 576 or
                                              (k <= 1280 and n > 32))
    for code in codes + [0x10400, 0x10403, 0x10404]:
        w.d.tile = code
        w.y.fill_(77)
        w.launch()
        got = w.y.cpu().numpy()
        np.testing.assert_array_equal(got[:m * n].reshape(m, n), want,
                                      err_msg=hex(code))
        assert (got[m * n:] == 77).all(), hex(code)
