"""Batch norm on small fp16 tensors, where the streaming passes add the partial sums themselves: at the edges of the slab of
channels, of the number of partial rows either side takes, and of the row groups of a block; and the sums of the block's row
lanes for every width of the channel vectors."""
import ctypes as C

import numpy as np
import pytest
import torch

from oracle import ref
from saga_amd import kernels as K
from tests.gpu_util import assert_close, dev, host, rnd

pytestmark = pytest.mark.gpu
HALF, F32 = torch.float16, torch.float32


# N, C, H, W, partial rows handed to the forward and the linked backward pass
@pytest.mark.parametrize("N,Cc,H,W,prows", [(1, 8, 1, 1, 1), (3, 16, 33, 31, 512), (3, 16, 33, 31, 513), (2, 24, 9, 11, 7), (2, 40, 9, 7, 33),
                                            (5, 64, 12, 11, 128), (5, 64, 12, 11, 129), (4, 72, 16, 16, 64), (7, 136, 13, 13, 65),
                                            (2, 512, 7, 7, 5), (1, 1032, 5, 3, 2), (9, 256, 25, 25, 57)])
@pytest.mark.parametrize("add", [0, 1])
def test_norm(N, Cc, H, W, prows, add):
    rng = np.random.default_rng(Cc + prows)
    L, stream = K.lib(), K.stream_ptr()
    x, z, dy = (rnd(rng, N, Cc, H, W, dtype=HALF) for _ in range(3))
    f = lambda a: np.asarray(a, np.float32)
    s, b, rm, rv = f(1 + 0.2 * rng.standard_normal(Cc)), f(0.1 * rng.standard_normal(Cc)), f(rng.standard_normal(Cc)), f(np.ones(Cc))
    flags = K.BN_RELU | (K.BN_ADD if add else 0)
    y, sm, si, nrm, nrv = ref.bn_train_fwd(x, s, b, rm, rv, 1e-3, 0.25)
    y = np.maximum(y + z if add else y, 0)
    flat = x.transpose(0, 2, 3, 1).reshape(-1, Cc).astype(np.float64)
    of = np.arange(len(flat)) % prows
    sums = lambda v: np.stack([v[of == p].sum(0) for p in range(prows)])
    partial = lambda u, v: dev(f(np.stack([sums(u), sums(v)], axis=2)))
    xd, zd, dyd = (dev(t, HALF, "nhwc") for t in (x, z, dy))
    yd = dev(np.full(x.shape, np.nan, np.float32), HALF, "nhwc")
    sd, bd, rmd, rvd, smd, sid = (dev(t) for t in (s, b, rm, rv, np.zeros(Cc, np.float32), np.zeros(Cc, np.float32)))
    vx, vz, vy, vdy = (K.view(t) for t in (xd, zd, yd, dyd))
    ws = torch.empty(L.saga_hip_bn_workspace_size(C.byref(vx)), dtype=torch.uint8, device="cuda")
    pd = partial(flat, flat * flat)
    K.check(L.saga_hip_bn_train_fwd_partials(C.byref(vx), C.byref(vz) if add else None, C.byref(vy), K.ptr(sd), K.ptr(bd), K.ptr(rmd),
                                             K.ptr(rvd), K.ptr(smd), K.ptr(sid), 1e-3, 0.25, flags, K.ptr(pd), prows, None, K.ptr(ws),
                                             ws.numel(), stream))
    assert_close(host(yd), y, HALF, "y", 4e-3)
    for got, want, what in ((smd, sm, "mean"), (sid, si, "1/std"), (rmd, nrm, "running mean"), (rvd, nrv, "running variance")):
        assert_close(host(got), want, F32, what, 1e-3)
    # backward, by itself and from the sums of a convolution
    yh = host(yd)
    g = dy * (yh > 0)
    dx, ds, db = ref.bn_bwd(x, g, s, host(smd), host(sid))
    for linked in ((0, 1) if not add else (0,)):
        dxd, dzd = (dev(np.full(x.shape, np.nan, np.float32), HALF, "nhwc") for _ in range(2))
        dsd, dbd = dev(np.ones(Cc, np.float32)), dev(np.ones(Cc, np.float32))
        vdx, vdz = K.view(dxd), K.view(dzd)
        if linked:
            gd = dev(g, HALF, "nhwc")
            vg = K.view(gd)
            gf = g.transpose(0, 2, 3, 1).reshape(-1, Cc).astype(np.float64)
            pg = partial(gf, gf * (flat - host(smd)))
            K.check(L.saga_hip_bn_bwd_linked(C.byref(vx), C.byref(vg), C.byref(vdx), K.ptr(sd), K.ptr(smd), K.ptr(sid), K.ptr(dsd), K.ptr(dbd),
                                             0.0, 1.0, K.ptr(pg), prows, K.ptr(ws), ws.numel(), stream))
        else:
            K.check(L.saga_hip_bn_bwd_ex(C.byref(vx), C.byref(vy), C.byref(vdy), C.byref(vdx), C.byref(vdz) if add else None, K.ptr(sd),
                                         K.ptr(bd), K.ptr(smd), K.ptr(sid), K.ptr(dsd), K.ptr(dbd), 0.0, 0.0, 1.0, flags, None, K.ptr(ws),
                                         ws.numel(), stream))
        scale = max(np.abs(ds).max(), np.abs(db).max(), 1.0)
        assert np.abs(host(dsd) - ds - 1).max() <= 2e-3 * scale and np.abs(host(dbd) - db - 1).max() <= 2e-3 * scale
        assert np.abs(host(dxd) - dx).max() <= 4e-3 * max(np.abs(dx).max(), 1.0)
        if add:
            np.testing.assert_array_equal(host(dzd), g)
