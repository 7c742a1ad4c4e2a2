"""Gradients with less workspace than their fastest kernels would use: the results are those of the oracle."""
import ctypes as C

import numpy as np
import pytest
import torch

from oracle import ref
from saga_amd import kernels as K
from tests.gpu_util import assert_close, dev, empty_like_layout, host, rnd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k,padc", [(21, 0), (24, 4)])
@pytest.mark.parametrize("share", [0, 0.5, 1])
def test_fp16_gradients_with_an_odd_pitch(k, padc, share):
    rng, dt = np.random.default_rng(1), torch.float16
    x, w = rnd(rng, 4, 16, 30, 30, dtype=dt), rnd(rng, k, 16, 3, 3, dtype=dt, scale=1 / 12)
    dy = rnd(rng, 4, k, 30, 30, dtype=dt)
    L, p, st = K.lib(), K.ConvParams(1, 1, 1, 1), K.stream_ptr()
    xd, wd, dyd = dev(x, dt, "nhwc"), dev(w, dt, "nhwc"), dev(dy, dt, "nhwc", padc)
    dx, dw = empty_like_layout(x.shape, dt, "nhwc"), empty_like_layout(w.shape, dt, "nhwc")
    vx, vw, vy = K.view(xd), K.view(wd), K.view(dyd)

    def room(kind):
        n = int(share * L.saga_hip_conv2d_workspace_size(kind, C.byref(vx), C.byref(vw), C.byref(vy), C.byref(p)))
        return (torch.empty(n, dtype=torch.uint8, device="cuda") if n else None), n

    ws, n = room(K.CONV_BWD_DATA)
    K.check(L.saga_hip_conv2d_bwd_data(C.byref(vy), C.byref(vw), C.byref(K.view(dx)), C.byref(p), 1.0, 0.0, K.ptr(ws), n, st))
    ws2, n = room(K.CONV_BWD_FILTER)
    K.check(L.saga_hip_conv2d_bwd_filter(C.byref(vx), C.byref(vy), C.byref(K.view(dw)), C.byref(p), 1.0, 0.0, K.ptr(ws2), n, st))
    torch.cuda.synchronize()
    assert_close(host(dx), ref.conv2d_bwd_data(dy, w, x.shape, 1, 1), dt, "dx", tol=2e-3)
    assert_close(host(dw), ref.conv2d_bwd_filter(x, dy, w.shape, 1, 1), dt, "dw", tol=2e-3)


# (c, k, r, stride): channels in eights and not, filters that are packed and that are read in place, residue classes
F32 = [(16, 24, 3, 1), (16, 24, 3, 2), (24, 16, 1, 1), (16, 8, 1, 2), (8, 40, 5, 1), (7, 13, 3, 1)]


@pytest.mark.parametrize("share", [0.3, 0.6, 1])
@pytest.mark.parametrize("c,k,r,stride", F32)
def test_fp32_convolutions(c, k, r, stride, share):
    rng, dt = np.random.default_rng(1), torch.float32
    pad = r // 2
    x, w = rnd(rng, 4, c, 30, 30), rnd(rng, k, c, r, r, scale=1 / np.sqrt(c * r * r))
    want = ref.conv2d_fwd(x, w, pad, stride)
    dy = rnd(rng, *want.shape)
    L, p, st = K.lib(), K.ConvParams(pad, stride, 1, 1), K.stream_ptr()
    xd, wd, dyd = dev(x), dev(w), dev(dy)
    y, dx, dw = (torch.empty_like(t) for t in (dyd, xd, wd))
    vx, vw, vdy, vy, vdx, vdw = (K.view(t) for t in (xd, wd, dyd, y, dx, dw))
    r_ = C.byref

    def call(kind, fn, a, b, out):
        """With the least whole kilobyte from `share` of the query's answer up that is accepted."""
        n = L.saga_hip_conv2d_workspace_size(kind, r_(vx), r_(vw), r_(vdy), r_(p))
        room = int(share * n) & ~1023
        while True:
            ws = torch.empty(max(room, 16), dtype=torch.uint8, device="cuda")
            rc = fn(r_(a), r_(b), r_(out), r_(p), 1.0, 0.0, K.ptr(ws), room, st)
            if rc != -4 or room > n:
                break
            room += 1024
        K.check(rc)

    call(K.CONV_FWD, L.saga_hip_conv2d_fwd, vx, vw, vy)
    call(K.CONV_BWD_DATA, L.saga_hip_conv2d_bwd_data, vdy, vw, vdx)
    call(K.CONV_BWD_FILTER, L.saga_hip_conv2d_bwd_filter, vx, vdy, vdw)
    torch.cuda.synchronize()
    # sums of up to 3600 products in fp32: rounding of some 1e-6 of the largest
    assert_close(host(y), want, dt, "y", tol=1e-5)
    assert_close(host(dx), ref.conv2d_bwd_data(dy, w, x.shape, pad, stride), dt, "dx", tol=1e-5)
    assert_close(host(dw), ref.conv2d_bwd_filter(x, dy, w.shape, pad, stride), dt, "dw", tol=1e-5)
