"""The staged large-GEMM blocks (64 x 128, 128 x 128, 256 x 128, 256 x 256)
against 64-bit integers: one row or column past and short of a block, and K of
one step up to more steps than the deepest ring has stages."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n", [
    (1, 16, 1), (63, 64, 127), (65, 128, 129), (127, 192, 96),
    (128, 256, 128), (129, 320, 131), (255, 336, 257), (256, 384, 256),
    (257, 448, 255), (512, 576, 512), (300, 1040, 70), (1025, 640, 260)])
def test_staged_blocks_bit_exact(hip, m, k, n):
    import torch

    from quantanything_amd.workloads import GemmWorkload

    w = GemmWorkload(seed=m + n, M=m, K=k, N=n)
    w.y = torch.full((m * n + 64,), 77, dtype=torch.int8, device="cuda")
    w.d.y = w.y.data_ptr()
    g = w.spec
    acc = (g["a"].astype(np.int64) - g["zp_in"]) @ g["w"].astype(np.int64)
    t = 31 + g["shift"]
    q = ((acc + g["bias"]) * g["mult"] + (1 << (t - 1))) >> t
    want = (np.clip(q + g["zp_out"], g["qmin"], g["qmax"]) - 128)
    for code in (0, 0x10400, 0x10403, 0x10404, 0x10410, 0x10411, 0x10412):
        w.d.tile = code
        w.y.fill_(77)
        w.launch()
        got = w.y.cpu().numpy()
        np.testing.assert_array_equal(got[:m * n].reshape(m, n), want,
                                      err_msg=hex(code))
        assert (got[m * n:] == 77).all(), hex(code)


@pytest.mark.parametrize("frag", [True, False])
@pytest.mark.parametrize("m,k,n", [
    (1, 1536, 2048), (63, 640, 2100), (64, 640, 2100), (40, 4096, 1000),
    (1030, 576, 1156), (10049, 32, 140), (12000, 64, 260)])
def test_default_choice_bit_exact(hip, m, k, n, frag):
    """Sizes on each side of the lines between the tiles, the narrow kernel
    and the blocks, without a tile code, with and without the weights in
    fragment order."""
    from quantanything_amd.workloads import GemmWorkload

    w = GemmWorkload(seed=m + n, M=m, K=k, N=n)
    if not frag:
        w.d.w_frag = None
    g = w.spec
    acc = ((g["a"].astype(np.float64) - g["zp_in"]) @
           g["w"].astype(np.float64)).astype(np.int64)  # exact below 2^53
    t = 31 + g["shift"]
    q = ((acc + g["bias"]) * g["mult"] + (1 << (t - 1))) >> t
    want = (np.clip(q + g["zp_out"], g["qmin"], g["qmax"]) - 128)
    w.launch()
    got = w.y.cpu().numpy()
    np.testing.assert_array_equal(got.reshape(m, n), want)


@pytest.mark.parametrize("m,k,n", [
    (1020, 256, 260), (1023, 384, 384), (1024, 384, 384), (197, 64, 1028),
    (600, 448, 512), (3000, 448, 64), (3000, 512, 64)])
def test_default_choice_with_a_residual(hip, m, k, n):
    """The same lines for products with a residual, whose blocks pay later."""
    import torch

    from quantanything_amd.workloads import GemmWorkload

    w = GemmWorkload(seed=m + n, M=m, K=k, N=n)
    g, d = w.spec, w.d
    r = np.random.default_rng(m).integers(-128, 128, (m, n)).astype(np.int8)
    rd = torch.from_numpy(r).cuda()
    d.res, d.res_sn, d.res_sc, d.res_so = rd.data_ptr(), n, 1, 128
    d.za, d.ma, d.sa = 128, 1 << 30, -1  # both operands as they are
    d.zb, d.mb, d.sb = 128, 1 << 30, -1
    d.add_sign, d.add_zp, d.add_qmax = 1, 128, 255
    w._plan(d, g["mult"], g["shift"], g["bias"])
    acc = (g["a"].astype(np.int64) - g["zp_in"]) @ g["w"].astype(np.int64)
    t = 31 + g["shift"]
    q = ((acc + g["bias"]) * g["mult"] + (1 << (t - 1))) >> t
    q = np.clip(q + g["zp_out"], g["qmin"], g["qmax"])
    want = np.clip((q - 128) + r + 128, 0, 255) - 128
    w.launch()
    np.testing.assert_array_equal(w.y.cpu().numpy().reshape(m, n), want)
