"""The fp32 forward convolutions of one to four input channels (csrc/thin_f32.hip): held to the kernel's forms on the stub
runtime; on the GPU against 64 bits, and with operands that have no three bf16 parts."""
import ctypes as C

import numpy as np
import pytest
import torch

from saga_amd import kernels as K
from tests import stub_gpu
from tests.gpu_util import dev, host, rnd
from tests.stub_gpu import on_stub

F32 = torch.float32

# N, C, H, W, K, R, stride, pad, dilation: channels of a block in 32s, wavefronts
SHAPES = {
    (3, 1, 28, 27, 20, 5, 1, 0, 1): (1, 4),
    (2, 3, 33, 35, 70, 3, 2, 1, 1): (2, 4),        # a ragged second block of channels
    (5, 2, 9, 7, 33, 1, 3, 0, 1): (2, 4),          # several images to a tile; rows and columns that no pixel sees
    (9000, 1, 6, 6, 4, 3, 1, 2, 2): (1, 8),        # more padding than image, dilation; blocks that walk several tiles
    (1, 4, 40, 301, 32, 3, 1, 1, 1): (1, 8),       # long rows
    (3, 3, 224, 230, 64, 7, 2, 3, 1): (2, 8),      # a long filter
    (9, 4, 63, 62, 8, 8, 1, 3, 1): (1, 8),         # as many reduction indices as there are
}


def call(shape, x, w, y, bias=None, stream=None):
    e = K.ConvExtras(bias=C.pointer(bias), relu=1) if bias is not None else K.ConvExtras()
    K.check(K.lib().saga_hip_conv2d_fwd_ex(C.byref(x), C.byref(w), C.byref(y), C.byref(K.ConvParams(shape[7], shape[6], shape[8], 1)), 0.0,
                                           C.byref(e), None, 0, stream))


def out_shape(shape):
    n, c, h, wd, k, r, stride, pad, dil = shape
    return n, k, *(1 + (s + 2 * pad - (r - 1) * dil - 1) // stride for s in (h, wd))


@on_stub
def test_shapes_are_what_they_are_said_to_be():
    for shape, want in SHAPES.items():
        n, c, h, wd, k, r = shape[:6]
        views = []
        for a, d in ((1 << 20, (n, c, h, wd)), (1 << 33, (k, c, r, r)), (1 << 34, out_shape(shape))):
            v = K.TensorView()
            v.ptr, v.dtype = a, K.FLOAT
            v.dims[:], v.strides[:] = d, [d[1] * d[2] * d[3], d[2] * d[3], d[3], 1]
            views.append(v)
        stub_gpu.launched()
        call(shape, *views)
        ((name, tile, blocks, threads),) = stub_gpu.launched()
        assert (name, tile[:2], threads) == ("stream_f32_k_thin", want, 64 * want[1]), (shape, name, tile)


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["nchw", "nhwc"])
@pytest.mark.parametrize("shape", SHAPES)
def test_against_64_bits(shape, layout):
    n, c, h, wd, k, r, stride, pad, dil = shape
    rng = np.random.default_rng(sum(shape))
    x, w, b = rnd(rng, n, c, h, wd, dtype=F32), rnd(rng, k, c, r, r, dtype=F32, scale=(2.0 / (c * r * r)) ** 0.5), rnd(rng, k, dtype=F32)
    conv = lambda bias: torch.nn.functional.conv2d(torch.from_numpy(x).double(), torch.from_numpy(w).double(), bias, stride, pad, dil)
    # six products per sixteen reduction indices, each rounding the sum by at most half a last place, at random
    bound = 2.0 ** -23 * (6 * max(c * r * r, 16) / 16) ** 0.5
    xd, wd_, bd = dev(x, F32, layout), dev(w, F32, layout), dev(b, F32).view(1, k, 1, 1)
    for bias in (None, K.view(bd)):
        want = conv(None if bias is None else torch.from_numpy(b).double())
        want = (want if bias is None else want.relu()).numpy()
        yd = dev(np.full(out_shape(shape), np.nan, np.float32), F32, layout)
        call(shape, K.view(xd), K.view(wd_), K.view(yd), bias, K.stream_ptr())
        got = host(yd).astype(np.float64)
        assert np.linalg.norm(got - want) <= bound * np.linalg.norm(want)


def plain(shape, x, w):
    """Of float32 operands on the host: the kernel's result."""
    yd = dev(np.full(out_shape(shape), 7.0, np.float32), F32)
    xd, wd = dev(x, F32), dev(w, F32)
    call(shape, K.view(xd), K.view(wd), K.view(yd), None, K.stream_ptr())
    return host(yd).astype(np.float64)


def reference(shape, x, w):
    return torch.nn.functional.conv2d(*(torch.from_numpy(a).double() for a in (x, w)), None, shape[6], shape[7], shape[8]).numpy()


@pytest.mark.gpu
@pytest.mark.parametrize("scales", [(-120, 80), (80, -120), (-140, 100), (-20, -100)], ids=str)
@pytest.mark.parametrize("shape", SHAPES)
def test_small_numbers(shape, scales):
    """Operands whose low bits a bf16 cannot hold, subnormal ones among them, are multiplied with all their bits."""
    n, c, h, wd, k, r, stride, pad, dil = shape
    rng = np.random.default_rng(2)
    x, w = rnd(rng, n, c, h, wd, dtype=F32), rnd(rng, k, c, r, r, dtype=F32, scale=(2.0 / (c * r * r)) ** 0.5)
    x, w = np.ldexp(x, scales[0]), np.ldexp(w, scales[1])
    want = reference(shape, x, w)
    bound = 2.0 ** -23 * (6 * max(c * r * r, 16) / 16) ** 0.5  # (as above)
    assert np.linalg.norm(plain(shape, x, w) - want) <= bound * np.linalg.norm(want)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES)
def test_numbers_without_three_parts(shape):
    """Infinities, NaNs and numbers next to the largest: where they belong, nowhere else; and what shares a wavefront with them is
    multiplied with all bits of its weights."""
    n, c, h, wd, k, r, stride, pad, dil = shape
    rng = np.random.default_rng(1)
    x, w = rnd(rng, n, c, h, wd, dtype=F32), rnd(rng, k, c, r, r, dtype=F32, scale=(2.0 / (c * r * r)) ** 0.5)
    for value in (np.inf, -np.inf, np.nan, 3.4e38):
        x.reshape(-1)[rng.integers(x.size)] = value
    w.reshape(-1)[rng.integers(w.size)] = 1.2345678e32
    want, spread = reference(shape, x, w), reference(shape, x.astype(np.float64) ** 2, w.astype(np.float64) ** 2)
    with np.errstate(over="ignore"):
        ref = want.astype(np.float32)
    got = plain(shape, x, w)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(ref))
    np.testing.assert_array_equal(got[np.isinf(ref)], ref[np.isinf(ref)])
    ok = np.isfinite(ref)
    # The largest of up to 10^7 errors, each a chain of roundings of up to half a unit at random: 2**-24 / sqrt(3) of a partial sum each,
    # which grows like the root of its length to the sum's deviation, or to the sum itself where that is larger.  (Weights without their
    # third part: some 2e-6 of a deviation on average.)
    size = np.sqrt(spread[ok]) + np.abs(want[ok])
    assert (np.abs(got[ok] - want[ok]) <= 6 * (2.0 ** -24 / 3 ** 0.5 * (c * r * r / 2) ** 0.5 + 2.0 ** -24) * size).all()
