"""The byte-split tile codes offered for a 16-bit layer name each kernel once
(host side: the descriptors point nowhere)."""

import ctypes

import pytest

from quantanything_amd import native
from quantanything_amd.executor import ConvDesc, DeviceExecutor

pytestmark = pytest.mark.skipif(not native.available(),
                                reason="library not built")


def _desc(cin, cout, k=3, y_sp=None, x_off=0):
    lib = native.library()
    cs = 4 if cin <= 4 else cin
    y_sp = y_sp or cout
    d = ConvDesc()
    d.x, d.x_code = 0x10000 + 2 * x_off, 2
    d.x_sn, d.x_sc, d.x_sp, d.x_add = 20 * 20 * cs, 1, cs, 3
    (d.N, d.C, d.H, d.W, d.Cout, d.KH, d.KW, d.SH, d.SW, d.PH, d.PW, d.DH,
     d.DW, d.G, d.OH, d.OW) = (2, cin, 20, 20, cout, k, k, 1, 1, k // 2,
                               k // 2, 1, 1, 1, 20, 20)
    ck, rows = ctypes.c_int64(0), ctypes.c_int64(0)
    lib.qa_pack_weights_f64_size(cout, cin, k, k, 1, ctypes.byref(ck),
                                 ctypes.byref(rows))
    d.w, d.w_code, d.w_layout = 0x20000, 8, 2
    d.w_kgp, d.w_rows, d.wide = ck.value, rows.value, 1
    d.mult = d.shift = 0x30000
    d.qmin, d.qmax = -32768, 32767
    d.y, d.y_code = 0x40000, 2
    d.y_sn, d.y_sc, d.y_sp = 400 * y_sp, 1, y_sp
    d.wsplit, d.wsplit_k = 0x50000, 0x60000
    return d


ALL = {0x11011, 0x11012, 0x11014, 0x11021, 0x11022, 0x11024}


@pytest.mark.parametrize("desc,kind,codes", [
    (dict(cin=32, cout=64), 1, {0x11011, 0x11012, 0x11014}),
    (dict(cin=32, cout=32), 1, {0x11011, 0x11012}),
    (dict(cin=3, cout=64), 2, {0x11011}),
    (dict(cin=32, cout=64, y_sp=66), 0, ALL),   # outputs off 8 bytes
    (dict(cin=576, cout=64), 0, ALL),           # weights past the LDS
    (dict(cin=32, cout=64, x_off=4), 0, ALL)])  # input off 16 bytes
def test_each_kernel_once(desc, kind, codes):
    d = _desc(**desc)
    assert native.library().qa_conv_split_lds(ctypes.byref(d)) == kind
    got = DeviceExecutor.tile_candidates(d)
    assert len(got) == len(set(got)) and got[0] == 0
    assert {c for c in got if c & 0x1000} == codes
