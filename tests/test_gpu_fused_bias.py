"""Bias (and relu) in the epilogues: convolutions, transposed convolutions, matrix products and poolings, one shape per kernel
that takes them along and one where a pass of its own follows."""
import ctypes as C

import numpy as np
import pytest
import torch

from oracle import ref
from saga_amd import api as S
from saga_amd import kernels as K
from saga_amd import networks as N
from tests.gpu_util import assert_close, dev, host, rnd

pytestmark = pytest.mark.gpu
HALF, F32 = torch.float16, torch.float32


def workspace(kind, x, w, y, p):
    n = K.lib().saga_hip_conv2d_workspace_size(kind, C.byref(x), C.byref(w), C.byref(y), C.byref(p))
    return torch.empty(max(n, 1), dtype=torch.uint8, device="cuda"), n


def layout(dtype):
    return "nhwc" if dtype == HALF else "nchw"


# N, C, H, W, K, R, stride, pad, relu
CONVS = {
    "fp16 small grid": (HALF, 2, 64, 9, 11, 40, 3, 1, 1, 0),
    "fp16 larger tile of a small grid": (HALF, 1, 720, 29, 28, 480, 3, 1, 1, 0),
    "fp16 shared tiles": (HALF, 1, 1048, 8, 7, 1048, 5, 1, 2, 0),
    "fp16 tiles of 128 channels": (HALF, 8, 32, 91, 90, 136, 3, 1, 1, 0),
    "fp16 tiles of 64 channels": (HALF, 8, 64, 97, 94, 12, 1, 1, 0, 0),
    "fp16 tiles of 64 channels (3x3)": (HALF, 32, 64, 56, 56, 64, 3, 1, 1, 0),
    "fp16 rows": (HALF, 40, 64, 56, 56, 64, 3, 1, 1, 0),
    "fp16 thin": (HALF, 2, 3, 40, 41, 24, 7, 2, 3, 0),
    "fp16 relu": (HALF, 2, 16, 9, 9, 8, 3, 1, 1, 1),
    "fp32 stream": (F32, 2, 24, 11, 13, 40, 3, 2, 1, 1),
    "fp32 table": (F32, 3, 1, 28, 28, 20, 5, 1, 0, 0),
    "fp32 tiles": (F32, 8, 8, 190, 191, 80, 1, 1, 0, 1),
}


@pytest.mark.parametrize("name", CONVS)
def test_convolution(name):
    dtype, N, Cc, H, W, Kk, R, stride, pad, relu = CONVS[name]
    rng = np.random.default_rng(Cc + H)
    x, b = rnd(rng, N, Cc, H, W, dtype=dtype), rnd(rng, Kk, dtype=dtype)
    w = rnd(rng, Kk, Cc, R, R, dtype=dtype, scale=(2.0 / (Cc * R * R)) ** 0.5)
    want = ref.conv2d_fwd(x, w, pad, stride) + b[None, :, None, None]
    if relu:
        want = np.maximum(want, 0)
    lay = layout(dtype)
    xd, wd, bd = dev(x, dtype, lay), dev(w, dtype, lay), dev(b, dtype)
    yd = dev(np.full(want.shape, np.nan, np.float32), dtype, lay)
    vx, vw, vb, vy, p = K.view(xd), K.view(wd), K.view(bd.view(1, Kk, 1, 1)), K.view(yd), K.ConvParams(pad, stride, 1, 1)
    ws, n = workspace(K.CONV_FWD, vx, vw, vy, p)
    e = K.ConvExtras(bias=C.pointer(vb), relu=relu)
    K.check(K.lib().saga_hip_conv2d_fwd_ex(C.byref(vx), C.byref(vw), C.byref(vy), C.byref(p), 0.0, C.byref(e), K.ptr(ws), n,
                                           K.stream_ptr()))
    assert_close(host(yd), want, dtype, name, tol=2e-3 if dtype == HALF else None)


# N, C (of the result), H, W, K, R, stride, pad
TRANSPOSED = {
    "fp16 small grid": (HALF, 1, 64, 22, 24, 128, 2, 2, 0),
    "fp16 tiles": (HALF, 6, 64, 128, 130, 128, 2, 2, 0),
    "fp16 larger tile of a small grid": (HALF, 1, 512, 60, 59, 1024, 3, 2, 1),
    "fp16 shared tiles": (HALF, 1, 592, 40, 41, 1016, 3, 2, 1),
    "fp16 classes no tap reaches": (HALF, 2, 64, 90, 91, 64, 1, 2, 0),
    "fp32": (F32, 2, 24, 12, 13, 32, 2, 2, 0),
    "fp32 accumulating": (F32, 2, 8, 10, 9, 16, 3, 1, 1),
    "fp32 larger filter": (F32, 2, 24, 30, 31, 16, 9, 1, 4),
    "fp32 larger stride": (F32, 1, 72, 31, 32, 8, 5, 5, 0),
    "fp32 tiles": (F32, 8, 72, 182, 183, 8, 1, 1, 0),
}


@pytest.mark.parametrize("name", TRANSPOSED)
def test_transposed_convolution(name):
    dtype, N, Cc, H, W, Kk, R, stride, pad = TRANSPOSED[name]
    beta = 1.0 if "accumulating" in name else 0.0
    rng = np.random.default_rng(Cc + H)
    P, Q = 1 + (H + 2 * pad - R) // stride, 1 + (W + 2 * pad - R) // stride
    dy, b = rnd(rng, N, Kk, P, Q, dtype=dtype), rnd(rng, Cc, dtype=dtype)
    w = rnd(rng, Kk, Cc, R, R, dtype=dtype, scale=(2.0 / (Kk * R * R)) ** 0.5)
    want = ref.conv2d_bwd_data(dy, w, (N, Cc, H, W), pad, stride) + b[None, :, None, None] + beta
    lay = layout(dtype)
    dyd, wd, bd, dxd = dev(dy, dtype, lay), dev(w, dtype, lay), dev(b, dtype), dev(np.ones(want.shape, np.float32), dtype, lay)
    vy, vw, vb, vx, p = K.view(dyd), K.view(wd), K.view(bd.view(1, Cc, 1, 1)), K.view(dxd), K.ConvParams(pad, stride, 1, 1)
    ws, n = workspace(K.CONV_BWD_DATA, vx, vw, vy, p)
    K.check(K.lib().saga_hip_conv2d_bwd_data_bias(C.byref(vy), C.byref(vw), None, C.byref(vb), C.byref(vx), C.byref(p), beta, K.ptr(ws),
                                                  n, K.stream_ptr()))
    assert_close(host(dxd), want, dtype, name, tol=2e-3 if dtype == HALF else None)


@pytest.mark.parametrize("dtype,bdtype", [(HALF, HALF), (HALF, F32), (F32, F32)])
@pytest.mark.parametrize("relu", [0, 1])
@pytest.mark.parametrize("M,N,Kd", [(3, 70, 130), (64, 33, 9), (1100, 1030, 40)])
def test_product(M, N, Kd, relu, dtype, bdtype):
    rng = np.random.default_rng(M)
    A, B, b = rnd(rng, M, Kd, dtype=dtype), rnd(rng, Kd, N, dtype=dtype), rnd(rng, N, dtype=dtype)
    want = A.astype(np.float64) @ B + b
    Ad, Bd, bd, Cd = dev(A, dtype), dev(B, dtype), dev(b, bdtype), dev(np.full((M, N), np.nan, np.float32), dtype)
    code = {HALF: K.HALF, F32: K.FLOAT}
    K.check(K.lib().saga_hip_gemm_bias(0, 0, M, N, Kd, 1.0, K.ptr(Ad), Kd, K.ptr(Bd), N, 0.0, K.ptr(Cd), N, code[dtype], K.ptr(bd),
                                       code[bdtype], relu, K.stream_ptr()))
    assert_close(host(Cd), np.maximum(want, 0) if relu else want, dtype, "product", tol=1e-3 if dtype == HALF else None)


@pytest.mark.parametrize("mode,k,stride,pad", [("max", 2, 2, 0), ("max", 5, 2, 1), ("avg", 3, 2, 1)])
@pytest.mark.parametrize("dtype", [F32, HALF])
def test_pooling(mode, k, stride, pad, dtype):
    rng = np.random.default_rng(k)
    x = rnd(rng, 2, 7, 11, 12, dtype=dtype) - 1.0
    x[0, 1, 2, 3] = np.nan
    want = ref.maxpool_fwd(x, k, pad, stride) if mode == "max" else ref.avgpool_fwd(x, k, pad, stride)
    want = np.where(np.isnan(want), want, np.maximum(want, 0))
    xd, yd = dev(x, dtype), dev(np.zeros(want.shape, np.float32), dtype)
    K.check(K.lib().saga_hip_pool_fwd_relu(K.POOL_MAX if mode == "max" else K.POOL_AVG, C.byref(K.view(xd)), C.byref(K.view(yd)), k, pad,
                                           stride, K.stream_ptr()))
    np.testing.assert_allclose(host(yd), want, atol=2e-3 if dtype == HALF else 1e-6)


@pytest.mark.parametrize("step", [2, 5])
@pytest.mark.parametrize("name", ["fp16 small grid", "fp16 rows", "fp16 relu", "fp32 stream", "fp32 table"])
def test_bias_with_gaps(name, step):
    """A column of a matrix: read at its stride, in a pass of its own."""
    dtype, N, Cc, H, W, Kk, R, stride, pad, relu = CONVS[name]
    rng = np.random.default_rng(step)
    x, wide = rnd(rng, N, Cc, H, W, dtype=dtype), rnd(rng, Kk, step, dtype=dtype)
    w = rnd(rng, Kk, Cc, R, R, dtype=dtype, scale=(2.0 / (Cc * R * R)) ** 0.5)
    b = wide[:, 1]
    want = ref.conv2d_fwd(x, w, pad, stride) + b[None, :, None, None]
    lay = layout(dtype)
    xd, wd, bd = dev(x, dtype, lay), dev(w, dtype, lay), dev(wide, dtype)[:, 1]
    yd = dev(np.full(want.shape, np.nan, np.float32), dtype, lay)
    vx, vw, vb, vy, p = K.view(xd), K.view(wd), K.view(bd), K.view(yd), K.ConvParams(pad, stride, 1, 1)
    assert list(vb.dims) == [Kk, 1, 1, 1] and vb.strides[0] == step
    L, st = K.lib(), K.stream_ptr()
    ws, n = workspace(K.CONV_FWD, vx, vw, vy, p)
    e = K.ConvExtras(bias=C.pointer(vb), relu=relu)
    K.check(L.saga_hip_conv2d_fwd_ex(C.byref(vx), C.byref(vw), C.byref(vy), C.byref(p), 0.0, C.byref(e), K.ptr(ws), n, st))
    assert_close(host(yd), np.maximum(want, 0) if relu else want, dtype, name, tol=2e-3 if dtype == HALF else None)
    if stride == 1:  # backward data of the same filter, with a bias per input channel
        wide = rnd(rng, step, Cc, dtype=dtype).T.copy()
        bd = dev(wide, dtype)[:, 0]
        vb = K.view(bd)
        ws, n = workspace(K.CONV_BWD_DATA, vx, vw, vy, p)
        dy = rnd(rng, *want.shape, dtype=dtype)
        dyd, dx = dev(dy, dtype, lay), dev(np.full(x.shape, np.nan, np.float32), dtype, lay)
        K.check(L.saga_hip_conv2d_bwd_data_bias(C.byref(K.view(dyd)), C.byref(vw), None, C.byref(vb), C.byref(K.view(dx)), C.byref(p),
                                                0.0, K.ptr(ws), n, st))
        want = ref.conv2d_bwd_data(dy, w, x.shape, pad, stride) + wide[:, 0][None, :, None, None]
        assert_close(host(dx), want, dtype, name + " transposed", tol=2e-3 if dtype == HALF else None)


@pytest.mark.parametrize("dtype", [S.FLOAT, S.HALF], ids=["f32", "f16"])
def test_bias_from_a_window(dtype):
    """The same in a program: convolution and product with a column of a matrix as their bias."""
    rng = np.random.default_rng(7)
    draw = lambda *shape: rng.standard_normal(shape).astype(N.np_dtype(dtype))
    x, w, m = draw(2, 8, 6, 6), draw(16, 8, 3, 3), draw(16, 3)
    fx, fw, fm = draw(4, 24), draw(24, 16), draw(16, 3)

    def column(g, a):
        return g.add_node("window", {"x": S.Tensor.from_numpy(a)}, {"offset": [0, 1], "shape": [16, 1]}).y()

    g = S.Graph()
    y = g.add_node("conv", {"x": S.Tensor.from_numpy(x), "w": S.Tensor.from_numpy(w), "b": column(g, m)},
                   {"size": 3, "activations": 16, "pad": 1, "bias": True}).y()
    f = g.add_node("fc", {"x": S.Tensor.from_numpy(fx), "w": S.Tensor.from_numpy(fw), "b": column(g, fm)},
                   {"outputs": 16, "bias": True}).y()
    ctx = S.Context()
    p = ctx.create_program(g, 2, training=False)
    y, f = ctx.resolve(y), ctx.resolve(f)
    p.run(1)
    tol = 2e-3 if dtype == S.HALF else 1e-5
    wide = lambda a: a.astype(np.float32)
    assert_close(wide(y.read()), ref.conv2d_fwd(wide(x), wide(w), 1, 1) + wide(m)[None, :, 1, None, None], None, "conv", tol=tol)
    assert_close(wide(f.read()), wide(fx) @ wide(fw) + wide(fm)[None, :, 1], None, "fc", tol=tol)
