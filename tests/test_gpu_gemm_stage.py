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


def _workload(m, k, n, res, y2, offset, images=None):
    """A GEMM (or the pointwise convolution over m / images pixels an image)
    with a residual, a rescaled copy in wider rows and weights past int8, its
    buffers and the values both outputs must hold."""
    import torch

    from quantanything_amd.utils import multiply_by_quantized_multiplier
    from quantanything_amd.workloads import GemmWorkload

    w = GemmWorkload(seed=m + n, M=m, K=k, N=n)
    g, d = w.spec, w.d
    rng = np.random.default_rng(m * n + k)
    wt = g["w"].astype(np.int32)
    if offset:  # each channel spans 255 values, none of them int8's
        wt = wt // 2 + rng.integers(-150, 151, (1, n)).astype(np.int32)
        d.w_kgp, d.w_rows, d.needs_rowsum = w._pack(
            np.ascontiguousarray(wt.T).reshape(n, k, 1, 1), int(d.x_add))
        assert d.needs_rowsum == 1
        d.w, d.corr, d.boff = (w.wp.data_ptr(), w.corr.data_ptr(),
                               w.boff.data_ptr())
    w.y = torch.full((m * n + 64,), 77, dtype=torch.int8, device="cuda")
    d.y = w.y.data_ptr()
    acc = ((g["a"].astype(np.float64) - g["zp_in"]) @
           wt.astype(np.float64)).astype(np.int64)  # exact below 2^53
    t = 31 + g["shift"]
    q = ((acc + g["bias"]) * g["mult"] + (1 << (t - 1))) >> t
    q = np.clip(q + g["zp_out"], g["qmin"], g["qmax"])
    if res:
        r = rng.integers(-128, 128, (m, n)).astype(np.int8)
        w.r = torch.from_numpy(r).cuda()
        d.res, d.res_sc, d.res_so = w.r.data_ptr(), 1, 128
        d.res_sn, d.res_sp = n, 0
        d.za, d.ma, d.sa = 128, 1 << 30, -1  # both operands as they are
        d.zb, d.mb, d.sb = 128, 1 << 30, -1
        d.add_sign, d.add_zp, d.add_qmax = 1, 128, 255
        q = np.clip((q - 128) + r + 128, 0, 255)
    want, want2 = q - 128, None
    if y2:
        w.y2 = torch.full((m * (n + 5) + 64,), 77, dtype=torch.int8,
                          device="cuda")
        d.y2, d.y2_sc, d.y2_sn, d.y2_sp = w.y2.data_ptr() + 3, 1, n + 5, 0
        d.r2_zp_in, d.r2_m, d.r2_s, d.r2_zp_out = 120, 1500000000, 0, 7
        d.r2_qmin, d.r2_qmax = 0, 255
        want2 = np.clip(multiply_by_quantized_multiplier(
            q.astype(np.int64) - 120, 1500000000, 0) + 7, 0, 255) - 128
    if images:
        hw = m // images
        d.N, d.H, d.W, d.OH, d.OW = images, 1, hw, 1, hw
        d.x_sn, d.x_sp, d.y_sn, d.y_sp = hw * k, k, hw * n, n
        if res:
            d.res_sn, d.res_sp = hw * n, n
        if y2:
            d.y2_sn, d.y2_sp = hw * (n + 5), n + 5
    w._plan(d, g["mult"], g["shift"], g["bias"])
    return w, want, want2


def _check(w, want, want2, m, n, what):
    w.y.fill_(77)
    if want2 is not None:
        w.y2.fill_(77)
    w.launch()
    got = w.y.cpu().numpy()
    np.testing.assert_array_equal(got[:m * n].reshape(m, n), want,
                                  err_msg=what)
    assert (got[m * n:] == 77).all(), what
    if want2 is not None:
        flat = w.y2.cpu().numpy()
        rows = flat[3:3 + m * (n + 5)].reshape(m, n + 5)
        np.testing.assert_array_equal(rows[:, :n], want2, err_msg=what)
        rows[:, :n] = 77
        assert (flat == 77).all(), what


@pytest.mark.parametrize("res", [False, True])
@pytest.mark.parametrize("y2", [False, True])
@pytest.mark.parametrize("offset", [False, True])
@pytest.mark.parametrize("m,k,n", [(257, 448, 259), (512, 256, 512),
                                   (130, 80, 97)])
def test_every_epilogue_form(hip, m, k, n, res, y2, offset):
    """Every block with a residual, a rescaled copy and weight offsets, on
    whole blocks and past them (256 x 256 has no residual or offset: 256 x
    128 then)."""
    w, want, want2 = _workload(m, k, n, res, y2, offset)
    for code in (0, 0x10400, 0x10403, 0x10404, 0x10410, 0x10411, 0x10412):
        w.d.tile = code
        _check(w, want, want2, m, n, hex(code))


@pytest.mark.parametrize("images,hw,k,n,res,y2,offset", [
    (4, 2116, 64, 128, False, True, False),     # 64 x 128 blocks
    (3, 4801, 96, 260, True, False, True),      # 128 x 128
    (4, 7056, 64, 512, False, True, False),     # 256 x 256
    (4, 7056, 64, 512, False, False, False),
    (2, 7056, 1024, 512, True, True, False),    # 256 x 128
    (2, 7056, 1024, 512, False, True, True)])
def test_pointwise_convolutions_as_gemms(hip, images, hw, k, n, res, y2,
                                         offset):
    """Pointwise convolutions past the narrow kernel's line, whose pixels are
    the rows of a GEMM on blocks that the library chooses."""
    m = images * hw
    # past the narrow kernel: no residual, blocks of 16 rows x 64 channels
    assert res or -(-m // 16) * -(-n // 64) > 1024
    w, want, want2 = _workload(m, k, n, res, y2, offset, images)
    _check(w, want, want2, m, n, "")
