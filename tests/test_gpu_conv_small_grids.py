"""fp16 convolutions whose grid of full tiles does not fill the chip: one shape per tile and split of the reduction that the
launch rules of csrc/stream_f16.hip and of the shared tiles in csrc/conv_mfma.hip choose, with remainders on every axis;
forward with its statistics and its folded norm, backward data with accumulation and with the link to a batch norm."""
import ctypes as C

import numpy as np
import pytest
import torch

from oracle import ref
from saga_amd import kernels as K
from tests.gpu_util import assert_close, dev, host, rnd

pytestmark = pytest.mark.gpu
HALF = torch.float16

# N, C, H, W, K, R, stride, pad.  The names say what the rules choose, forward and, where it is something else, backward
# (tests/test_kernel_routes.py holds them to it): pixels x channels of a wavefront's tile and what the block's wavefronts share.
SHAPES = {
    "16x16, four along the pixels": (1, 80, 10, 11, 24, 1, 1, 0),
    "16x16, four along the reduction": (1, 136, 5, 4, 152, 1, 1, 0),
    "16x16, four along the reduction (3x3)": (1, 400, 5, 6, 72, 3, 1, 1),
    "16x16, four along the reduction (whole slices)": (1, 256, 6, 7, 40, 3, 1, 1),
    "16x16, four along the reduction; backward 16x16, four along the pixels": (2, 512, 5, 5, 24, 1, 1, 0),
    "16x16, four along the reduction; backward 16x16, four along the pixels (three images)": (3, 256, 9, 9, 64, 1, 1, 0),
    "32x32, two and two": (1, 176, 69, 70, 56, 1, 1, 0),
    "32x32, four along the reduction": (1, 104, 27, 26, 168, 1, 1, 0),
    "32x32, four along the reduction; backward 16x16, four along the reduction": (2, 64, 30, 31, 128, 3, 1, 1),
    "32x32, four along the reduction (3x3)": (4, 256, 14, 13, 248, 3, 1, 1),
    "64x32, two and two": (5, 72, 45, 44, 80, 3, 1, 1),
    "64x32, eight along the reduction": (3, 232, 22, 24, 232, 1, 1, 0),
    "64x32, eight along the reduction (3x3)": (8, 384, 7, 13, 512, 3, 1, 1),
    "64x64, two and two": (5, 464, 24, 23, 488, 1, 1, 0),
    "64x64, four along the reduction": (1, 488, 38, 40, 496, 1, 1, 0),
    "64x64, four along the reduction (3x3)": (1, 256, 50, 53, 256, 3, 1, 1),
    "64x64, four along the reduction; backward 32x32, four along the reduction": (1, 72, 50, 53, 256, 3, 1, 1),
    "16x16, four along the reduction; backward classes of 32x32, four along the reduction": (3, 64, 19, 17, 48, 3, 2, 1),
    "16x16, four along the pixels; backward classes, some that no tap reaches, of 16x16, four along the pixels": (2, 64, 11, 12, 64, 1, 2, 0),
    "64x64, four along the reduction; backward classes of 64x64, two and two": (1, 512, 60, 59, 1024, 3, 2, 1),
    "shared 256x128 tiles": (1, 1048, 8, 7, 1048, 5, 1, 2),
    "shared 256x64 tiles; backward 256x128 tiles": (1, 816, 66, 65, 40, 3, 1, 1),
    "backward shared 256x64 tiles": (5, 48, 40, 41, 760, 3, 1, 1),
    "backward classes of shared 256x128 tiles": (1, 592, 40, 41, 1016, 3, 2, 1),
    "64x32, eight along the reduction; backward 64x64, four along the reduction": (1, 720, 29, 28, 480, 3, 1, 1),
    "64x64, four along the reduction; backward 256x128 tiles": (1, 256, 120, 122, 64, 3, 1, 1),
    "32x32, four along the reduction; backward classes of 64x32, eight along the reduction": (3, 168, 21, 23, 240, 1, 2, 0),
    "256x64 tiles": (3, 48, 70, 71, 48, 1, 1, 0),
    "256x128 tiles": (5, 112, 45, 47, 112, 1, 1, 0),
}


def params(rng, n):
    f = lambda a: np.asarray(a, np.float32)
    return (f(1 + 0.3 * rng.standard_normal(n)), f(0.2 * rng.standard_normal(n)), f(0.1 * rng.standard_normal(n)),
            f(rng.uniform(0.5, 1.5, n)))


@pytest.mark.parametrize("name", SHAPES)
def test_forward(name):
    N, Cc, H, W, Kk, R, stride, pad = SHAPES[name]
    rng = np.random.default_rng(Cc + H)
    L, S = K.lib(), K.stream_ptr()
    x = rnd(rng, N, Cc, H, W, dtype=HALF)
    w = rnd(rng, Kk, Cc, R, R, dtype=HALF, scale=(2.0 / (Cc * R * R)) ** 0.5)
    want = ref.conv2d_fwd(x, w, pad, stride)
    xd, wd, yd = dev(x, HALF, "nhwc"), dev(w, HALF, "nhwc"), dev(np.full(want.shape, 9.0, np.float32), HALF, "nhwc")
    p = K.ConvParams(pad, stride, 1, 1)
    vx, vw, vy = K.view(xd), K.view(wd), K.view(yd)
    ws = K._ws(L.saga_hip_conv2d_workspace_size(K.CONV_FWD, C.byref(vx), C.byref(vw), C.byref(vy), C.byref(p)), xd)
    # statistics: the stored outputs' own sums
    nbytes = L.saga_hip_conv2d_fwd_bnstats_size(C.byref(vx), C.byref(vw), C.byref(vy), C.byref(p))
    part = torch.full((nbytes // 4,), float("nan"), device="cuda")
    rows = C.c_int(0)
    K.check(L.saga_hip_conv2d_fwd_bnstats(C.byref(vx), C.byref(vw), C.byref(vy), C.byref(p), 1.0, K.ptr(ws), ws.numel(),
                                          K.ptr(part), nbytes, C.byref(rows), S))
    assert_close(host(yd), want, HALF, "y")
    sums = host(part[: rows.value * Kk * 2].reshape(rows.value, Kk, 2)).astype(np.float64).sum(0)
    stored = host(yd).astype(np.float64)
    np.testing.assert_allclose(sums[:, 0], stored.sum((0, 2, 3)), rtol=1e-4, atol=1e-3 * np.abs(stored).max() * stored[0, 0].size ** 0.5)
    np.testing.assert_allclose(sums[:, 1], (stored ** 2).sum((0, 2, 3)), rtol=1e-4)
    # accumulation
    K.conv2d(K.CONV_FWD, xd, wd, yd, pad, stride, alpha=0.5, beta=1.0)
    assert_close(host(yd), 1.5 * want, HALF, "accumulated y")
    # the folded norm with a residual and relu
    s, b, m, v = params(rng, Kk)
    z = rnd(rng, *want.shape, dtype=HALF)
    zd, sd, bd, md, vd = dev(z, HALF, "nhwc"), dev(s), dev(b), dev(m), dev(v)
    K.check(L.saga_hip_conv2d_fwd_bn_infer(C.byref(vx), C.byref(vw), C.byref(vy), C.byref(K.view(zd)), C.byref(p), K.ptr(sd), K.ptr(bd),
                                           K.ptr(md), K.ptr(vd), 1e-5, K.BN_RELU | K.BN_ADD, K.ptr(ws), ws.numel(), S))
    r = lambda a: a.reshape(1, -1, 1, 1)
    sc = s / np.sqrt(v + 1e-5)
    assert_close(host(yd), np.maximum(want * r(sc) + r(b - m * sc) + z, 0), HALF, "folded norm")


@pytest.mark.parametrize("name", SHAPES)
def test_backward_data(name):
    N, Cc, H, W, Kk, R, stride, pad = SHAPES[name]
    rng = np.random.default_rng(Cc + W)
    L, S = K.lib(), K.stream_ptr()
    P, Q = 1 + (H + 2 * pad - R) // stride, 1 + (W + 2 * pad - R) // stride
    dy = rnd(rng, N, Kk, P, Q, dtype=HALF)
    w = rnd(rng, Kk, Cc, R, R, dtype=HALF, scale=(2.0 / (Kk * R * R)) ** 0.5)
    want = ref.conv2d_bwd_data(dy, w, (N, Cc, H, W), pad, stride)
    dyd, wd, dxd = dev(dy, HALF, "nhwc"), dev(w, HALF, "nhwc"), dev(np.full(want.shape, 9.0, np.float32), HALF, "nhwc")
    K.conv2d(K.CONV_BWD_DATA, dyd, wd, dxd, pad, stride)
    assert_close(host(dxd), want, HALF, "dx")
    plain = host(dxd)
    K.conv2d(K.CONV_BWD_DATA, dyd, wd, dxd, pad, stride, beta=1.0)
    assert_close(host(dxd), 2 * want, HALF, "accumulated dx")
    # linked to the backward of a norm + relu: the same gradient under the relu's mask, and its sums
    s, b, m, v = params(rng, Cc)
    x = rnd(rng, N, Cc, H, W, dtype=HALF)
    xd, sd, bd, md, vd = dev(x, HALF, "nhwc"), dev(s), dev(b), dev(m), dev(v)
    p = K.ConvParams(pad, stride, 1, 1)
    vdy, vw, vdx, vx = K.view(dyd), K.view(wd), K.view(dxd), K.view(xd)
    ws = K._ws(L.saga_hip_conv2d_workspace_size(K.CONV_BWD_DATA, C.byref(vdx), C.byref(vw), C.byref(vdy), C.byref(p)), xd)
    nbytes = L.saga_hip_conv2d_bwd_data_bnbwd_size(C.byref(vdy), C.byref(vw), C.byref(vdx), C.byref(p))
    assert nbytes > 0
    part = torch.full((nbytes // 4,), float("nan"), device="cuda")
    link = K.BnBwdLink(C.pointer(vx), K.ptr(sd), K.ptr(bd), K.ptr(md), K.ptr(vd), K.BN_RELU, 0, K.ptr(part), nbytes)
    K.check(L.saga_hip_conv2d_bwd_data_bnbwd(C.byref(vdy), C.byref(vw), None, C.byref(vdx), C.byref(p), 1.0, 0.0, K.ptr(ws),
                                             ws.numel(), C.byref(link), S))
    r = lambda a: a.reshape(1, -1, 1, 1)
    pre = x.astype(np.float64) * r(s * v) + r(b - m * s * v)
    got = host(dxd)
    keep = got != 0
    clear = np.abs(pre) > 1e-3  # (away from zero, where the order of roundings decides)
    np.testing.assert_array_equal(keep[clear], ((pre > 0) & (plain != 0))[clear])
    np.testing.assert_array_equal(got[keep], plain[keep])
    sums = host(part[: link.partial_rows * Cc * 2].reshape(link.partial_rows, Cc, 2)).astype(np.float64).sum(0)
    g = got.astype(np.float64)
    atol = 1e-3 * np.abs(g).max() * g[0, 0].size ** 0.5
    np.testing.assert_allclose(sums[:, 0], g.sum((0, 2, 3)), rtol=1e-4, atol=atol)
    np.testing.assert_allclose(sums[:, 1], (g * (x - r(m))).sum((0, 2, 3)), rtol=1e-4, atol=4 * atol)
