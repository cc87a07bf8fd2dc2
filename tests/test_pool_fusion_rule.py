"""The planner's choice between a convolution fused with its global average
pool and the two launches, at the measured sizes on each side of its lines
(host side)."""

import pytest

from quantanything_amd.executor import ConvDesc, DeviceExecutor


@pytest.mark.parametrize("n,cin,cout,size,k,fused", [
    (1, 128, 256, 14, 1, True), (1024, 128, 256, 7, 1, True),
    (32, 64, 64, 10, 3, True),  # small images
    (32, 64, 128, 20, 1, False), (64, 64, 128, 20, 1, True),
    (256, 64, 128, 20, 1, True),
    (32, 128, 256, 20, 1, False), (256, 128, 256, 20, 1, True),
    (1024, 128, 256, 20, 1, True),
    (16, 384, 1280, 10, 1, True), (32, 384, 1280, 10, 1, False),
    (64, 256, 512, 14, 1, True), (128, 256, 512, 14, 1, False),
    (256, 128, 256, 28, 1, False), (32, 128, 256, 56, 1, False),
    (32, 64, 64, 20, 3, False)])
def test_choice(n, cin, cout, size, k, fused):
    d = ConvDesc()
    (d.N, d.C, d.H, d.W, d.Cout, d.KH, d.KW, d.SH, d.SW, d.PH, d.PW, d.OH,
     d.OW) = n, cin, size, size, cout, k, k, 1, 1, k // 2, k // 2, size, size
    d.w_kgp = -(-cin * k * k // 64) * 4
    assert DeviceExecutor.pool_fusion_pays(d) == fused
