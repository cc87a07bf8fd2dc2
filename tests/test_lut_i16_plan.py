"""The LDS form of a 16-bit activation table (qa_plan_lut_i16, on the host)
decodes to the table, entry for entry, outside the groups its header names;
tables that are not smooth are refused."""

import ctypes

import numpy as np
import pytest

from quantanything_amd import native

pytestmark = pytest.mark.skipif(not native.available(),
                                reason="library not built")


def _plan(lut):
    lib = native.library()
    lut = np.ascontiguousarray(lut, np.int32)
    size = lib.qa_lut_i16_plan_bytes(len(lut))
    assert size == 16 + -(-(-(-len(lut) // 16) * 8) // 16) * 16
    plan = np.zeros(size, np.uint8)
    rc = lib.qa_plan_lut_i16(lut.ctypes.data, len(lut),
                             ctypes.c_void_p(plan.ctypes.data))
    return rc, plan


def _decode(plan, n):
    head = plan[:16].view(np.int32)
    w = plan[16:].view(np.uint32).astype(np.int64)
    i = np.arange(n)
    a, b, f = w[2 * (i >> 4)], w[2 * (i >> 4) + 1], i & 15
    k0, d = a & 0xFFFF, (a >> 16) - (a & 0xFFFF)
    v = head[0] + k0 + ((d * f + 8) >> 4) + ((b >> (2 * f)) & 3) - 2
    odd = np.isin(i >> 4, head[2:4])
    return v, odd


def _silu(n, scale, out, lo, hi):
    x = (np.arange(n) - n // 2) * scale
    return np.clip(np.rint(x / (1 + np.exp(-x)) / out), lo, hi).astype(
        np.int64)


@pytest.mark.parametrize("n", [1, 15, 16, 17, 4096, 40000, 65536])
@pytest.mark.parametrize("out", [2e-4, 1.3e-4])  # without and with clipping
def test_smooth_tables(n, out):
    lut = _silu(n, 1.6e-4, out, -32768, 32767)
    rc, plan = _plan(lut)
    assert rc == 1
    v, odd = _decode(plan, n)
    assert odd.sum() <= 32
    np.testing.assert_array_equal(v[~odd], lut[~odd])


def test_identity_offset_and_extremes():
    lut = np.arange(65536) + 2**30
    rc, plan = _plan(lut)
    v, odd = _decode(plan, 65536)
    assert rc == 1 and not odd.any()
    np.testing.assert_array_equal(v, lut)


def test_refused():
    rng = np.random.default_rng(1)
    assert _plan(rng.integers(-100, 100, 65536))[0] == 0
    assert _plan([0, 70000])[0] == 0
    lib = native.library()
    assert lib.qa_lut_i16_plan_bytes(0) == -1
    assert lib.qa_lut_i16_plan_bytes(65537) == -1
    assert lib.qa_plan_lut_i16(None, 5, None) == -1
