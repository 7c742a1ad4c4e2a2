"""Batch norm on channels-first tensors, whose channels are shared by several blocks: planes of whole vectors and of odd sizes, one
block to a channel and as many as one adds up, runs that end inside a plane, slices of wider tensors, addresses off the vectors'
alignment, results over the input."""
import ctypes as C

import numpy as np
import pytest
import torch

from oracle import ref
from saga_amd import kernels as K
from tests.gpu_util import assert_close, host, rnd

pytestmark = pytest.mark.gpu
HALF, F32 = torch.float16, torch.float32

# N, C, H, W, channels on either side in the tensor it is a slice of, elements before it
SHAPES = [(1, 2, 1, 2, 0, 0), (3, 5, 1, 4, 0, 0), (2, 3, 7, 9, 0, 0), (33, 16, 8, 8, 0, 0), (33, 16, 8, 8, 0, 1), (5, 70, 13, 12, 2, 0),
          (4, 6, 32, 32, 0, 0), (1, 4, 64, 64, 0, 0), (5, 3, 31, 33, 1, 0), (300, 2, 64, 64, 0, 0), (1025, 4, 3, 3, 0, 0), (2, 600, 4, 8, 0, 0)]


def placed(a, dtype, side, shift):
    """The array as a slice of a tensor of more channels, `shift` elements behind an aligned address."""
    n, c, h, w = a.shape
    flat = torch.zeros(n * (c + 2 * side) * h * w + shift, dtype=dtype, device="cuda")
    t = flat[shift:].view(n, c + 2 * side, h, w)[:, side:side + c]
    t.copy_(torch.from_numpy(a))
    return t


@pytest.mark.parametrize("dtype", [F32, HALF], ids=["f32", "f16"])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_planes(shape, dtype):
    N, Cc, H, W, side, shift = shape
    rng = np.random.default_rng(N + Cc)
    L, stream = K.lib(), K.stream_ptr()
    x, z, dy = (rnd(rng, N, Cc, H, W, dtype=dtype) for _ in range(3))
    x += 3 * rng.standard_normal(Cc).astype(np.float16).astype(np.float32).reshape(1, -1, 1, 1)
    x = x.astype(np.float16).astype(np.float32) if dtype == HALF else x
    f = lambda a: torch.from_numpy(np.asarray(a, np.float32)).cuda()
    s, b, rm, rv = 1 + 0.2 * rng.standard_normal(Cc), 0.1 * rng.standard_normal(Cc), rng.standard_normal(Cc), 0.5 + rng.random(Cc)
    s, b, rm, rv = (a.astype(np.float32) for a in (s, b, rm, rv))
    sd, bd, md, vd = f(s), f(b), f(rm), f(rv)
    put = lambda a: placed(a, dtype, side, shift)
    view = lambda t: C.byref(K.view(t))
    # inference
    xd, zd, yd = put(x), put(z), put(np.zeros_like(x))
    K.check(L.saga_hip_bn_infer(view(xd), view(zd), view(yd), K.ptr(sd), K.ptr(bd), K.ptr(md), K.ptr(vd), 1e-3, K.BN_ADD | K.BN_RELU, stream))
    assert_close(host(yd), np.maximum(ref.bn_infer(x, s, b, rm, rv, 1e-3) + z, 0), dtype, "inference")
    y0, sm, si, nrm, nrv = ref.bn_train_fwd(x, s, b, rm, rv, 1e-3, 0.25)
    for flags, in_place in ((0, 0), (K.BN_RELU, 1), (K.BN_RELU | K.BN_ADD, 0)):
        add = flags & K.BN_ADD
        rmd, rvd, smd, sid = f(rm), f(rv), f(rm), f(rm)
        xd, zd = put(x), put(z)
        yd = xd if in_place else put(np.zeros_like(x))
        ws = K.bn_workspace(xd)
        K.check(L.saga_hip_bn_train_fwd(view(xd), view(zd) if add else None, view(yd), K.ptr(sd), K.ptr(bd), K.ptr(rmd), K.ptr(rvd),
                                        K.ptr(smd), K.ptr(sid), 1e-3, 0.25, flags, K.ptr(ws), ws.numel(), stream))
        y = y0 + z if add else y0
        y = np.maximum(y, 0) if flags & K.BN_RELU else y
        assert_close(host(yd), y, dtype, "y")
        for got, want, what in ((smd, sm, "mean"), (sid, si, "1/std"), (rmd, nrm, "running mean"), (rvd, nrv, "running variance")):
            assert_close(host(got), want, F32, what)
        # backward; dx added to what was there, or over dy
        xd, yh = put(x), host(yd)
        g = dy * (yh > 0) if flags else dy
        dx, ds, db = ref.bn_bwd(x, g, s, host(smd), host(sid))
        dyd, dzd = put(dy), put(np.ones_like(x))
        dxd = dyd if in_place else put(np.ones_like(x))
        beta = 0.0 if in_place else 1.0
        for beta_dz in ((0.0, 1.0) if add else (0.0,)):
            dsd, dbd = f(np.ones(Cc)), f(np.ones(Cc))
            K.check(L.saga_hip_bn_bwd_ex(view(xd), view(yd), view(dyd), view(dxd), view(dzd) if add else None, K.ptr(sd), K.ptr(bd),
                                         K.ptr(smd), K.ptr(sid), K.ptr(dsd), K.ptr(dbd), beta, beta_dz, 1.0, flags, None, K.ptr(ws),
                                         ws.numel(), stream))
            scale = max(np.abs(ds).max(), np.abs(db).max(), 1.0)
            assert np.abs(host(dsd) - 1 - ds).max() <= 1e-4 * scale and np.abs(host(dbd) - 1 - db).max() <= 1e-4 * scale
            assert_close(host(dxd), dx * (1 + beta_dz) + beta, dtype, "dx")
            if add:
                np.testing.assert_array_equal(host(dzd), (g * (1 + beta_dz)).astype(np.float16).astype(np.float32) if dtype == HALF else g * (1 + beta_dz))


# a channel that its block does not quite hold between the sums and what follows (1025 vectors; fp16: 4100 values), and one that it
# just does (1024 values off the vectors' alignment)
@pytest.mark.parametrize("dtype", [F32, HALF], ids=["f32", "f16"])
@pytest.mark.parametrize("shape", [(41, 3, 10, 10, 0, 0), (16, 5, 8, 8, 0, 1)], ids=str)
def test_planes_at_what_a_block_holds(shape, dtype):
    test_planes(shape, dtype)
