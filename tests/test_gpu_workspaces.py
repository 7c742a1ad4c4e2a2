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
