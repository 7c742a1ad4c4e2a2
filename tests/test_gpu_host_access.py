"""Host access to device tensors: Tensor.write and Tensor.read move every element to its place and back, whatever the
layout of the device tensor, the size (staged, whole, sample by sample) and the number of channels."""
import ctypes

import numpy as np
import pytest
import torch

from saga_amd import api as S
from saga_amd import kernels as K

pytestmark = pytest.mark.gpu

# channels 1 .. 4 have loops of their own on the host, 64 is the width of a tile on the device; the last two are
# larger than the staging memory, one of them with samples larger than a chunk
SHAPES = [(1, 1, 1, 1), (2, 1, 5, 7), (3, 2, 4, 4), (1, 3, 33, 65), (2, 4, 9, 3), (2, 5, 17, 31), (1, 63, 3, 5), (2, 64, 8, 8),
          (3, 65, 1, 9), (5, 130, 7, 1), (70, 3, 96, 97), (2, 40, 331, 333)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("dtype", [S.HALF, S.FLOAT])
@pytest.mark.parametrize("batched", [False, True])
@pytest.mark.parametrize("layout", [S.LAYOUT_NHWC, S.LAYOUT_NCHW])
def test_write_and_read_back(shape, dtype, batched, layout):
    rng = np.random.default_rng(sum(shape))
    np_dt = np.float16 if dtype == S.HALF else np.float32

    def values():
        return rng.integers(1, 2000, shape).astype(np_dt)  # exact in both types, positive

    first = values()
    x = S.Tensor.from_numpy(first)
    g = S.Graph()
    y = g.add_node("relu", {"x": x}).y()
    ctx = S.Context()
    p = ctx.create_program(g, shape[0], training=False, tensor_layout=layout, batched={x: S.PRE} if batched else None)
    dx, dy = ctx.resolve(x), ctx.resolve(y)
    p.run(1)
    np.testing.assert_array_equal(dy.read(), first)
    for _ in range(3):
        v = values()
        dx.write(v)
        if not batched:
            np.testing.assert_array_equal(dx.read(), v)
        p.run(1)
        np.testing.assert_array_equal(dy.read(), v)
    # a run that nobody wrote for works on what was written last
    p.run(2)
    if not batched:
        np.testing.assert_array_equal(dy.read(), v)


@pytest.mark.parametrize("layout", [S.LAYOUT_NHWC, S.LAYOUT_NCHW])
def test_slices_of_a_wider_tensor(layout):
    """Inputs of a concat live in slices of its output: a write leaves the neighbours alone."""
    rng = np.random.default_rng(5)
    a, b = (rng.integers(1, 2000, (2, c, 6, 5)).astype(np.float16) for c in (3, 9))
    g = S.Graph()
    ta, tb = S.Tensor.from_numpy(a), S.Tensor.from_numpy(b)
    ra, rb = g.add_node("relu", {"x": ta}).y(), g.add_node("relu", {"x": tb}).y()
    y = g.add_node("concat", {"x0": ra, "x1": rb}, {"axis": 1}).y()
    ctx = S.Context()
    p = ctx.create_program(g, 2, training=False, tensor_layout=layout)
    da, db, dy = ctx.resolve(ra), ctx.resolve(rb), ctx.resolve(y)
    p.run(1)
    np.testing.assert_array_equal(da.read(), a)
    np.testing.assert_array_equal(db.read(), b)
    np.testing.assert_array_equal(dy.read(), np.concatenate([a, b], 1))
    da.write(a + 1)
    np.testing.assert_array_equal(da.read(), a + 1)
    np.testing.assert_array_equal(dy.read(), np.concatenate([a + 1, b], 1))


# the tile of a transposition is 64 channels by up to 1024 pixels; the third layout has none of its own
@pytest.mark.parametrize("shape", [(1, 1, 1, 1), (2, 3, 33, 65), (2, 64, 8, 8), (3, 65, 1, 9), (2, 130, 5, 13)])
@pytest.mark.parametrize("dtype", ["uint8", "int16", "int32", "int64"])
def test_copies_of_bit_patterns(shape, dtype):
    t = torch.from_numpy(np.random.default_rng(len(dtype)).integers(0, 256, shape).astype(dtype))
    t = (t * 127).cuda()
    n, c, h, w = shape

    def like(order):
        wide = torch.full((n, c, h, w) if order == "nchw" else (w, h, n, c + 1) if order == "whnc" else (n, h, w, c + (order == "slice")), 7,
                          dtype=t.dtype, device="cuda")
        return wide, {"nchw": lambda: wide, "nhwc": lambda: wide.permute(0, 3, 1, 2), "slice": lambda: wide[..., :c].permute(0, 3, 1, 2),
                      "whnc": lambda: wide[..., :c].permute(2, 3, 1, 0)}[order]()

    for a in ("nchw", "nhwc", "slice", "whnc"):
        for b in ("nchw", "nhwc", "slice", "whnc"):
            (_, src), (wide, dst) = like(a), like(b)
            src.copy_(t)
            K.check(K.lib().saga_hip_copy(ctypes.byref(K.view(src)), ctypes.byref(K.view(dst)), K.stream_ptr()))
            assert torch.equal(dst, t), (a, b)
            if b in ("slice", "whnc"):
                assert bool((wide[..., c] == 7).all()), (a, b)
