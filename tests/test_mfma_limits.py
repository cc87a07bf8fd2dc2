"""Layers past the int8 MFMA launches' 32-bit limits are not sent to them by
the executor (they keep the general path, which takes them)."""

import pytest

from quantanything_amd.executor import DeviceExecutor


def _geo(n=2, size=(9, 9), k=(3, 3), dil=(1, 1), out=(7, 7)):
    return (n, 24, *size, 24, *k, 1, 1, 0, 0, *dil, 24, *out)


@pytest.mark.parametrize("geo,ok", [
    (_geo(), True),
    (_geo(n=2**31 // 49), True), (_geo(n=2**31 // 49 + 1), False),
    (_geo(size=(70000, 9), k=(2, 3), dil=(32767, 1), out=(9, 7)), True),
    (_geo(size=(70000, 9), k=(2, 3), dil=(32768, 1), out=(9, 7)), False),
    (_geo(size=(9, 70000), k=(3, 3), dil=(1, 16384), out=(7, 9)), False),
    (_geo(n=2**31 - 1, size=(1, 1), k=(1, 1), out=(1, 1)), True),
    (_geo(n=2**31, size=(1, 1), k=(1, 1), out=(1, 1)), False)])
def test_limits(geo, ok):
    assert DeviceExecutor._mfma_limits(geo) == ok
