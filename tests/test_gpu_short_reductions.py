"""Reductions that few blocks or lanes would otherwise carry: the fully-connected product on small grids, averages over wide
windows, max-pool gradients of windows that tile a plane, bias gradients of planes, and the sums of filter-gradient
partials; at the edges of their tiles, vectors and lane counts."""
import ctypes as C

import numpy as np
import pytest
import torch

from oracle import ref
from saga_amd import kernels as K
from tests import test_gpu_ops as test_ops
from tests.gpu_util import assert_close, dev, host, rnd

pytestmark = pytest.mark.gpu
HALF, F32 = torch.float16, torch.float32


def S():
    return K.stream_ptr()


@pytest.mark.parametrize("tA", [0, 1])
@pytest.mark.parametrize("tB", [0, 1])
@pytest.mark.parametrize("M,N,Kd", [(1, 1000, 2048), (1, 1, 17), (33, 65, 67), (32, 32, 64), (40, 72, 520), (31, 70, 130),
                                    (64, 48, 4096), (520, 512, 128), (1000, 1024, 264)])
def test_gemm_split(M, N, Kd, tA, tB):
    rng = np.random.default_rng(M + Kd)
    A, B = rnd(rng, M, Kd, dtype=HALF), rnd(rng, Kd, N, dtype=HALF)
    Ad, Bd = dev(A.T if tA else A, HALF), dev(B.T if tB else B, HALF)
    Cd = dev(np.ones((M, N), np.float32), HALF)
    K.check(K.lib().saga_hip_gemm(tA, tB, M, N, Kd, 0.5, K.ptr(Ad), Ad.shape[1], K.ptr(Bd), Bd.shape[1], 1.0, K.ptr(Cd), N,
                                  K.HALF, S()))
    assert_close(host(Cd), 0.5 * (A.astype(np.float64) @ B) + 1, HALF, "gemm", tol=1e-3)


@pytest.mark.parametrize("tA", [0, 1])
@pytest.mark.parametrize("tB", [0, 1])
@pytest.mark.parametrize("M,N,Kd", [(1, 1, 1), (5, 3, 2), (16, 16, 32), (17, 33, 129), (64, 1024, 3136), (260, 250, 128), (250, 260, 131),
                                    (500, 512, 65), (512, 512, 512), (31, 1030, 64)])
def test_gemm_split_fp32(M, N, Kd, tA, tB):
    rng = np.random.default_rng(M + Kd)
    A, B = rnd(rng, M, Kd), rnd(rng, Kd, N)
    Ad, Bd = dev(A.T if tA else A), dev(B.T if tB else B)
    Cd = dev(np.ones((M, N), np.float32))
    K.check(K.lib().saga_hip_gemm(tA, tB, M, N, Kd, 0.5, K.ptr(Ad), Ad.shape[1], K.ptr(Bd), Bd.shape[1], 1.0, K.ptr(Cd), N,
                                  K.FLOAT, S()))
    assert_close(host(Cd), 0.5 * (A.astype(np.float64) @ B) + 1, F32, "gemm", tol=1e-5)


@pytest.mark.parametrize("layout,padc,dtype", [("nhwc", 0, HALF), ("nhwc", 8, HALF), ("nchw", 0, HALF), ("nchw", 0, F32), ("nhwc", 0, F32)])
@pytest.mark.parametrize("k,pad,stride,H", [(4, 0, 4, 9), (7, 0, 7, 7), (8, 3, 2, 12), (15, 0, 1, 15), (16, 0, 1, 17), (31, 2, 3, 33),
                                            (90, 0, 1, 90)])
def test_average_shared_by_lanes(k, pad, stride, H, layout, padc, dtype):
    rng = np.random.default_rng(k)
    x = rnd(rng, 3, 24, H, H, dtype=dtype)
    want = ref.avgpool_fwd(x, k, pad, stride)
    xd, yd = dev(x, dtype, layout, padc), dev(np.full(want.shape, 5.0, np.float32), dtype, layout, padc)
    K.check(K.lib().saga_hip_pool_fwd(K.POOL_AVG, C.byref(K.view(xd)), C.byref(K.view(yd)), None, k, pad, stride, S()))
    assert_close(host(yd), want, dtype, "avgpool", tol=1e-3 if dtype == HALF else 1e-5)


@pytest.mark.parametrize("dtype", [F32, HALF])
@pytest.mark.parametrize("beta", [0.0, 1.0])
@pytest.mark.parametrize("k,H,W", [(2, 8, 8), (2, 9, 11), (2, 3, 2), (3, 9, 9), (3, 10, 11), (3, 3, 5)])
def test_max_gradient_of_tiling_windows(k, H, W, beta, dtype):
    rng = np.random.default_rng(k + H)
    x = np.maximum(rnd(rng, 5, 7, H, W, dtype=dtype), 0)
    x[1, 2, 0, 1] = np.nan
    x[2, 3] = -np.inf
    y = ref.maxpool_fwd(x, k, 0, k, with_idx=True)[0]
    dy = rnd(rng, *y.shape, dtype=dtype)
    dxd = dev(np.ones(x.shape, np.float32), dtype)
    K.check(K.lib().saga_hip_pool_bwd(K.POOL_MAX, *(C.byref(K.view(t)) for t in (dev(x, dtype), dev(y, dtype), dev(dy, dtype), dxd)),
                                      k, 0, k, beta, S()))
    assert_close(host(dxd), ref.maxpool_bwd(x, dy, k, 0, k) + beta, dtype, "maxpool bwd", tol=1e-3 if beta else 1e-7)


@pytest.mark.parametrize("dtype", [F32, HALF])
@pytest.mark.parametrize("shape", [(64, 20, 24, 24), (1, 3, 1, 1), (5, 7, 13, 13), (3, 2, 64, 64), (2, 5, 65, 64)])
def test_bias_gradient_of_planes(shape, dtype):
    rng = np.random.default_rng(shape[0])
    y = rnd(rng, *shape, dtype=dtype)
    db = dev(np.ones(shape[1], np.float32))
    K.check(K.lib().saga_hip_bias_bwd(C.byref(K.view(dev(y, dtype))), C.byref(K.view(db.view(1, shape[1], 1, 1))), 1.0, None, 0, S()))
    scale = np.abs(y.astype(np.float64)).sum(axis=(0, 2, 3)).max()
    assert np.abs(host(db) - (ref.bias_bwd(y) + 1)).max() <= 2e-6 * scale + 1e-6


# the gradient in the tensor's own 16-bit type: 2**-10 of it is more than its rounding (channels-last, the last two: in two passes)
@pytest.mark.parametrize("layout,padc", [("nchw", 0), ("nhwc", 0), ("nhwc", 3)])
@pytest.mark.parametrize("shape", [(1, 3, 1, 1), (5, 7, 13, 13), (2, 64, 129, 65), (1, 67, 127, 126)])
def test_bias_gradient_of_16_bits(shape, layout, padc):
    rng = np.random.default_rng(shape[0])
    y = rnd(rng, *shape, dtype=HALF)
    yd, db = dev(y, HALF, layout, padc), dev(np.ones(shape[1], np.float32), HALF)
    yv = K.view(yd)
    room = K.lib().saga_hip_bias_bwd_workspace_size(C.byref(yv))
    assert (room > 0) == (layout == "nhwc" and y.size >= 1 << 20)
    ws = torch.empty(max(room, 4), dtype=torch.uint8, device="cuda")
    K.check(K.lib().saga_hip_bias_bwd(C.byref(yv), C.byref(K.view(db.view(1, shape[1], 1, 1))), 1.0, K.ptr(ws) if room else None, room, S()))
    want = ref.bias_bwd(y) + 1
    scale = np.abs(y.astype(np.float64)).sum(axis=(0, 2, 3)).max()
    assert (np.abs(host(db) - want) <= 2.0**-10 * np.abs(want) + 2e-6 * scale + 1e-6).all()


# few, some and many partials per element; channels that are padded to vectors (fp16) and tap-major columns (fp32, 32)
@pytest.mark.parametrize("dtype,layout", [(HALF, "nhwc"), (F32, "nchw"), (F32, "nhwc")])
@pytest.mark.parametrize("N,Cc,H,Kk", [(1, 3, 5, 7), (2, 5, 40, 24), (16, 3, 32, 16), (8, 32, 24, 20)])
def test_sum_of_filter_partials(N, Cc, H, Kk, dtype, layout):
    rng = np.random.default_rng(Cc + H)
    x, dy = rnd(rng, N, Cc, H, H, dtype=dtype), rnd(rng, N, Kk, H, H, dtype=dtype)
    want = ref.conv2d_bwd_filter(x, dy, (Kk, Cc, 3, 3), 1, 1)
    dw = dev(np.ones(want.shape, np.float32), dtype, layout)
    K.conv2d(K.CONV_BWD_FILTER, dev(x, dtype, layout), dev(dy, dtype, layout), dw, 1, 1, beta=1.0)
    assert_close(host(dw), want + 1, dtype, "bwd filter", tol=2e-3 if dtype == HALF else 1e-5)


@pytest.mark.parametrize("N,Cc,H,W,Kk,R,stride,pad", [(2, 16, 9, 7, 1, 1, 1, 0), (3, 24, 13, 11, 7, 3, 1, 1), (2, 3, 40, 33, 20, 7, 2, 3),
                                                      (2, 13, 21, 19, 39, 5, 2, 2), (4, 64, 56, 56, 60, 3, 1, 1), (1, 70, 30, 31, 202, 3, 4, 1)])
def test_fp16_gradients_of_other_channel_counts(N, Cc, H, W, Kk, R, stride, pad):
    """Output channels in other numbers than eights: dy goes through a padded copy."""
    rng = np.random.default_rng(Kk)
    x = rnd(rng, N, Cc, H, W, dtype=HALF)
    w = rnd(rng, Kk, Cc, R, R, dtype=HALF, scale=(2.0 / (Cc * R * R)) ** 0.5)
    P, Q = 1 + (H + 2 * pad - R) // stride, 1 + (W + 2 * pad - R) // stride
    dy = rnd(rng, N, Kk, P, Q, dtype=HALF)
    for padc in (0, 3):  # dense, and a slice of a wider tensor
        xd, wd, dyd = dev(x, HALF, "nhwc"), dev(w, HALF, "nhwc"), dev(dy, HALF, "nhwc", padc)
        dw, dx = dev(np.ones(w.shape, np.float32), HALF, "nhwc"), dev(np.ones(x.shape, np.float32), HALF, "nhwc")
        K.conv2d(K.CONV_BWD_FILTER, xd, dyd, dw, pad, stride, beta=1.0)
        assert_close(host(dw), ref.conv2d_bwd_filter(x, dy, w.shape, pad, stride) + 1, HALF, "dw", tol=2e-3)
        K.conv2d(K.CONV_BWD_DATA, dyd, wd, dx, pad, stride, beta=1.0)
        assert_close(host(dx), ref.conv2d_bwd_data(dy, w, x.shape, pad, stride) + 1, HALF, "dx", tol=2e-3)


@pytest.mark.parametrize("dtype", [HALF, F32])
@pytest.mark.parametrize("tA", [0, 1])
@pytest.mark.parametrize("tB", [0, 1])
@pytest.mark.parametrize("M,N,Kd", [(8, 8, 8), (9, 10, 15), (39, 10, 64), (64, 10, 1024), (35, 17, 9), (17, 35, 70), (4, 5, 131), (33, 66, 7)])
def test_gemm_runs(M, N, Kd, tA, tB, dtype):
    """Runs that end where an operand's row does, at any address: operands inside larger ones full of NaN."""
    rng = np.random.default_rng(M + N + Kd)
    A, B = rnd(rng, M, Kd, dtype=dtype), rnd(rng, Kd, N, dtype=dtype)

    def inside(a):
        t = torch.full((a.shape[0] + 2, a.shape[1] + 3), float("nan"), device="cuda", dtype=dtype)
        t[1:-1, 1:-2] = dev(a, dtype)
        return t, t.data_ptr() + (t.shape[1] + 1) * t.element_size()

    Ad, pa = inside(A.T if tA else A)
    Bd, pb = inside(B.T if tB else B)
    Cd = dev(np.ones((M, N), np.float32), dtype)
    K.check(K.lib().saga_hip_gemm(tA, tB, M, N, Kd, 0.5, pa, Ad.shape[1], pb, Bd.shape[1], 1.0, K.ptr(Cd), N,
                                  K.HALF if dtype == HALF else K.FLOAT, S()))
    assert_close(host(Cd), 0.5 * (A.astype(np.float64) @ B) + 1, dtype, "gemm", tol=1e-3 if dtype == HALF else 1e-5)


@pytest.mark.parametrize("dtype", [HALF, F32])
@pytest.mark.parametrize("H", [700, 1401, 2800, 5450])
def test_blocks_of_several_patch_rows(H, dtype):
    """Tall images, whose blocks walk 2 to 16 rows of patches, the last one fewer, in the passes of the norm's backward."""
    test_ops.test_batch_norm_backward_through_a_max_pooling(1, H, 9, True, 0.0, dtype)
