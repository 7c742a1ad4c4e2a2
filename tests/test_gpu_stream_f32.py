"""The fp32 matrix products that read their operands straight from memory (csrc/stream_f32.hip): one case per tile and per
split of the reduction that the launch rule can choose, at sizes with remainders on every axis, forward and backward data
against the oracle, and the GEMM's four operand orders with partial last steps."""
import ctypes as C

import numpy as np
import pytest
import torch

from oracle import ref
from saga_amd import kernels as K
from tests.gpu_util import assert_close, dev, host, rnd

pytestmark = pytest.mark.gpu
F32 = torch.float32

# N, C, H, W, K, R, stride, pad: what the launch rule chooses forward (tests/test_kernel_routes.py holds it to that)
CONVS = [
    # filters read in place or through the table
    (2, 8, 255, 257, 65, 1, 1, 0),    # 64x64 tiles, four along the pixels
    (1, 1032, 79, 80, 200, 1, 1, 0),  # 64x64 tiles, the reduction over four wavefronts
    (1, 392, 90, 92, 40, 1, 1, 0),    # 64x32 tiles, the reduction over four
    (1, 16, 311, 317, 7, 1, 1, 0),    # 64x32 tiles, four along the pixels
    (3, 64, 9, 7, 31, 1, 1, 0),       # 32x32, few steps per wavefront
    (2, 13, 12, 11, 9, 5, 2, 2),      # table: channels in other numbers than eights
    (1, 3, 23, 29, 16, 7, 2, 3),
    # packed filters
    (1, 24, 180, 183, 72, 3, 1, 1),   # 64x64 tiles, four along the pixels
    (1, 24, 311, 317, 24, 3, 1, 1),   # 64x32 tiles, four along the pixels
    (1, 40, 157, 158, 64, 3, 1, 1),   # 32x32, four along the pixels
    (1, 16, 141, 142, 64, 3, 1, 1),   # 32x32, two and two
    (1, 128, 150, 161, 64, 3, 1, 1),  # 32x32, the reduction over four
    (1, 48, 127, 131, 30, 3, 1, 1),
    (1, 512, 3, 5, 33, 3, 1, 1),      # 32x32, sixteen wavefronts along the reduction
    (2, 24, 11, 13, 40, 3, 2, 1),     # residue classes backward
    (2, 16, 10, 9, 24, 2, 3, 0),      # stride beyond the filter: classes no tap reaches
    (2, 8, 9, 9, 8, 3, 4, 1),
]

# beside that kernel: tiles in LDS, forward or (more than 48 input channels, few output channels) backward, and filters of more
# taps and strides of more classes than it takes
LDS = [(5, 13, 182, 183, 72, 1, 1, 0), (9, 8, 182, 183, 56, 3, 1, 1), (8, 72, 182, 183, 8, 1, 1, 0), (8, 56, 182, 183, 8, 3, 1, 1),
       (2, 8, 30, 31, 72, 9, 1, 4), (1, 72, 40, 41, 20, 9, 2, 4), (2, 16, 31, 33, 24, 3, 5, 1), (1, 70, 26, 27, 9, 2, 5, 0)]


@pytest.mark.parametrize("shape", CONVS + LDS)
@pytest.mark.parametrize("layout", ["nchw", "nhwc"])
def test_conv(shape, layout):
    N, Cc, H, W, Kk, R, stride, pad = shape
    rng = np.random.default_rng(sum(shape))
    x = rnd(rng, N, Cc, H, W, dtype=F32)
    w = rnd(rng, Kk, Cc, R, R, dtype=F32, scale=(2.0 / (Cc * R * R)) ** 0.5)
    y_ref = ref.conv2d_fwd(x, w, pad, stride)
    dy = rnd(rng, *y_ref.shape, dtype=F32)
    xd, wd, dyd = dev(x, F32, layout), dev(w, F32, layout), dev(dy, F32, layout)
    yd = dev(np.full(y_ref.shape, 7.0, np.float32), F32, layout)
    K.conv2d(K.CONV_FWD, xd, wd, yd, pad, stride)
    assert_close(host(yd), y_ref, F32, "y")
    K.conv2d(K.CONV_FWD, xd, wd, yd, pad, stride, alpha=0.5, beta=1.0)
    assert_close(host(yd), 1.5 * y_ref, F32, "accumulated y")
    dxd = dev(np.full(x.shape, 7.0, np.float32), F32, layout)
    K.conv2d(K.CONV_BWD_DATA, dyd, wd, dxd, pad, stride)
    dx_ref = ref.conv2d_bwd_data(dy, w, x.shape, pad, stride)
    assert_close(host(dxd), dx_ref, F32, "dx")
    K.conv2d(K.CONV_BWD_DATA, dyd, wd, dxd, pad, stride, alpha=0.5, beta=1.0)
    assert_close(host(dxd), 1.5 * dx_ref, F32, "accumulated dx")


@pytest.mark.parametrize("tA,tB", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("size", [(64, 1030, 400), (33, 31, 17), (1, 1, 24), (5, 70, 1027), (130, 300, 65), (640, 2048, 20),
                                  # 64x64 tiles without and with a split, 64x32 tiles without and with; a reduction for the LDS tiles
                                  (2890, 3010, 21), (1300, 1290, 1030), (1000, 3100, 20), (520, 1060, 390), (640, 1030, 9)])
def test_gemm(tA, tB, size):
    M, N, Kd = size
    rng = np.random.default_rng(M + N + Kd)
    A, B = rnd(rng, M, Kd, dtype=F32), rnd(rng, Kd, N, dtype=F32)
    want = A.astype(np.float64) @ B.astype(np.float64)
    Ad, Bd = dev(A.T if tA else A, F32), dev(B.T if tB else B, F32)
    Cd = dev(np.ones((M, N), np.float32), F32)
    stream = K.stream_ptr()
    K.check(K.lib().saga_hip_gemm(tA, tB, M, N, Kd, 2.0, K.ptr(Ad), Ad.shape[1], K.ptr(Bd), Bd.shape[1], 3.0, K.ptr(Cd), N,
                                  K.FLOAT, stream))
    assert_close(host(Cd), 2 * want + 3, F32, "C")
    K.check(K.lib().saga_hip_gemm(tA, tB, M, N, Kd, 1.0, K.ptr(Ad), Ad.shape[1], K.ptr(Bd), Bd.shape[1], 0.0, K.ptr(Cd), N,
                                  K.FLOAT, stream))
    assert_close(host(Cd), want, F32, "C, overwritten")


@pytest.mark.parametrize("flags", [0, K.BN_RELU, K.BN_ADD | K.BN_RELU])
@pytest.mark.parametrize("shape", CONVS + LDS + [(8, 8, 190, 191, 80, 1, 1, 0), (2, 3, 186, 184, 64, 3, 1, 1)])
def test_folded_norm(shape, flags):
    N, Cc, H, W, Kk, R, stride, pad = shape
    rng = np.random.default_rng(sum(shape) + flags)
    x = rnd(rng, N, Cc, H, W, dtype=F32)
    w = rnd(rng, Kk, Cc, R, R, dtype=F32, scale=(2.0 / (Cc * R * R)) ** 0.5)
    f = lambda a: np.asarray(a, np.float32)
    s, b = f(1 + 0.3 * rng.standard_normal(Kk)), f(0.2 * rng.standard_normal(Kk))
    m, v = f(0.1 * rng.standard_normal(Kk)), f(rng.uniform(0.5, 1.5, Kk))
    y = ref.conv2d_fwd(x, w, pad, stride)
    z = rnd(rng, *y.shape, dtype=F32)
    col = lambda a: a[None, :, None, None]
    want = (y - col(m)) * col(s / np.sqrt(v + 1e-3)) + col(b)
    if flags & K.BN_ADD:
        want = want + z
    if flags & K.BN_RELU:
        want = np.maximum(want, 0)
    xd, wd, zd = dev(x, F32), dev(w, F32), dev(z, F32, "nhwc")
    yd = dev(np.full(y.shape, np.nan, np.float32), F32)
    L, p = K.lib(), K.ConvParams(pad, stride, 1, 1)
    vx, vw, vy, vz = (K.view(t) for t in (xd, wd, yd, zd))
    n = L.saga_hip_conv2d_workspace_size(K.CONV_FWD, C.byref(vx), C.byref(vw), C.byref(vy), C.byref(p))
    ws = torch.empty(max(n, 1), dtype=torch.uint8, device="cuda")
    prm = [dev(a, F32) for a in (s, b, m, v)]
    K.check(L.saga_hip_conv2d_fwd_bn_infer(C.byref(vx), C.byref(vw), C.byref(vy), C.byref(vz) if flags & K.BN_ADD else None,
                                           C.byref(p), *(K.ptr(t) for t in prm), 1e-3, flags, K.ptr(ws), n, K.stream_ptr()))
    assert_close(host(yd), want, F32, "folded norm")


@pytest.mark.parametrize("shape", CONVS + [(3, 64, 150, 161, 64, 1, 1, 0)])
def test_packed_filter(shape):
    """Forward and backward data from a filter that was packed beforehand: the same results as packing per call gives."""
    N, Cc, H, W, Kk, R, stride, pad = shape
    rng = np.random.default_rng(sum(shape))
    x = rnd(rng, N, Cc, H, W, dtype=F32)
    w = rnd(rng, Kk, Cc, R, R, dtype=F32, scale=(2.0 / (Cc * R * R)) ** 0.5)
    y = ref.conv2d_fwd(x, w, pad, stride)
    dy = rnd(rng, *y.shape, dtype=F32)
    L, p, stream = K.lib(), K.ConvParams(pad, stride, 1, 1), K.stream_ptr()
    xd, wd, dyd = dev(x, F32), dev(w, F32), dev(dy, F32)
    for kind, want in ((K.CONV_FWD, y), (K.CONV_BWD_DATA, ref.conv2d_bwd_data(dy, w, x.shape, pad, stride))):
        out = dev(np.full(want.shape, np.nan, np.float32), F32)
        vx, vw, vy = (K.view(t) for t in ((xd, wd, out) if kind == K.CONV_FWD else (out, wd, dyd)))
        args = (kind, C.byref(vx), C.byref(vw), C.byref(vy), C.byref(p))
        n = L.saga_hip_conv2d_pack_bytes(*args)
        assert (n > 0) == ((Cc if kind == K.CONV_FWD else Kk) % 8 == 0)
        if not n:
            continue
        packed = torch.full((n // 4,), np.nan, device="cuda")
        jobs = (K.FilterPackJob * 16)()
        count = L.saga_hip_conv2d_pack_jobs(*args, K.ptr(packed), jobs)
        blocks = 0
        for j in jobs[:count]:
            j.first_block = blocks
            blocks += j.blocks
        table = torch.frombuffer(bytearray(C.string_at(jobs, C.sizeof(K.FilterPackJob) * count)), dtype=torch.uint8).cuda()
        K.check(L.saga_hip_filter_pack_batched(K.ptr(table), count, blocks, stream))
        if kind == K.CONV_FWD:
            e = K.ConvExtras(packed=packed.data_ptr())
            K.check(L.saga_hip_conv2d_fwd_ex(C.byref(vx), C.byref(vw), C.byref(vy), C.byref(p), 0.0, C.byref(e), None, 0, stream))
        else:
            K.check(L.saga_hip_conv2d_bwd_data_wt(C.byref(vy), C.byref(vw), K.ptr(packed), C.byref(vx), C.byref(p), 1.0, 0.0, None, 0,
                                                  stream))
        assert_close(host(out), want, F32, "packed")
