"""The fp32 convolutions that stage windows of the input (csrc/window_f32.hip): one shape per form of launch, held to it on the
stub runtime; on the GPU against 64 bits, and with operands that have no three bf16 parts."""
import ctypes as C

import numpy as np
import pytest
import torch

from saga_amd import kernels as K
from tests import stub_gpu
from tests.gpu_util import dev, host, rnd
from tests.stub_gpu import on_stub

F32 = torch.float32

# N, C, H, W, K, R, stride, pad: forward launch's tile rows in 32s, rounds of loads, taps, wavefronts
SHAPES = {
    (3, 48, 17, 11, 33, 1, 1, 0): (1, 2, 1, 1),      # images of no whole fours, a ragged last tile of both kinds
    (70, 200, 16, 16, 170, 1, 1, 0): (2, 1, 1, 8),   # three whole slices and one of eight channels
    (9, 136, 27, 30, 72, 1, 2, 0): (1, 4, 1, 2),     # pixels apart
    (40, 64, 43, 64, 170, 1, 3, 0): (1, 1, 1, 8),
    (90, 56, 33, 32, 96, 1, 2, 1): (1, 1, 1, 4),     # some of them outside the image
    (9, 104, 7, 7, 40, 3, 1, 1): (1, 1, 9, 4),       # windows over several images; half a step of channels
    (8, 64, 28, 30, 128, 3, 1, 1): (2, 1, 9, 8),     # the reduction over four
    (5, 40, 70, 66, 64, 3, 1, 1): (2, 1, 9, 4),      # 128 pixels to a window
    (7, 24, 20, 126, 17, 3, 1, 1): (1, 2, 9, 4),     # two rounds of loads
    (60, 24, 21, 23, 40, 3, 2, 1): (1, 1, 9, 4),     # stride 2 (backward: classes, not here)
    (4, 64, 14, 14, 64, 5, 1, 2): (1, 1, 25, 4),     # the reduction over four
    (60, 16, 28, 28, 130, 5, 1, 0): (1, 1, 25, 4),   # backward: more padding than the filter needs, pixels out of order: not here
}

# straight from memory (csrc/stream_f32.hip): backward residue classes of pixels, of filters as they are; and, too few pixels for a
# window, filters in three parts
CLASSES, FEW = (2, 24, 11, 13, 40, 3, 2, 1), (1, 24, 9, 11, 40, 3, 1, 1)


def views(shape, x, w, y):
    """Views of dense tensors at these addresses."""
    n, c, h, wd, k, r, stride, pad = shape
    out = []
    for a, d in ((x, (n, c, h, wd)), (w, (k, c, r, r)), (y, (n, k, 1 + (h + 2 * pad - r) // stride, 1 + (wd + 2 * pad - r) // stride))):
        v = K.TensorView()
        v.ptr, v.dtype = a, K.FLOAT
        v.dims[:], v.strides[:] = d, [d[1] * d[2] * d[3], d[2] * d[3], d[3], 1]
        out.append(v)
    return out


def run(kind, shape, x, w, y, packed, beta=0.0):
    """The convolution from a packed filter, as a program runs it (a call of its own packs no small 1x1 filters)."""
    vx, vw, vy = (C.byref(v) for v in views(shape, x, w, y))
    p, L = C.byref(K.ConvParams(shape[7], shape[6], 1, 1)), K.lib()
    if kind == K.CONV_FWD:
        K.check(L.saga_hip_conv2d_fwd_ex(vx, vw, vy, p, beta, C.byref(K.ConvExtras(packed=packed)), None, 0, None))
    else:
        K.check(L.saga_hip_conv2d_bwd_data_wt(vy, vw, packed, vx, p, 1.0, beta, None, 0, None))


@on_stub
def test_shapes_are_what_they_are_said_to_be():
    for shape, (tm, rounds, taps, waves) in SHAPES.items():
        stub_gpu.launched()
        run(K.CONV_FWD, shape, 1 << 20, 1 << 33, 1 << 34, 1 << 35)
        ((name, tile, blocks, threads),) = stub_gpu.launched()
        assert name == "stream_f32_k_window" and (tile[0], tile[3], tile[4], threads) == (tm, rounds, taps, 64 * waves), (shape, tile, threads)


@on_stub
def test_packed_filters_without_windows():
    for shape, kind, q in ((CLASSES, K.CONV_FWD, 4), (CLASSES, K.CONV_BWD_DATA, 3), (FEW, K.CONV_FWD, 4), (FEW, K.CONV_BWD_DATA, 4)):
        stub_gpu.launched()
        run(kind, shape, 1 << 20, 1 << 33, 1 << 34, 1 << 35)
        ((name, tile, blocks, threads),) = stub_gpu.launched()
        assert (name, tile[1]) == ("stream_f32_k", q), (shape, kind, tile)


def reference(shape, x, w, dy):
    n, c, h, wd, k, r, stride, pad = shape
    x = torch.from_numpy(x).double().requires_grad_()
    y = torch.nn.functional.conv2d(x, torch.from_numpy(w).double(), None, stride, pad)
    y.backward(torch.from_numpy(dy).double())
    return y.detach().numpy(), x.grad.numpy()


def operands(shape):
    n, c, h, wd, k, r, stride, pad = shape
    rng = np.random.default_rng(sum(shape))
    x = rnd(rng, n, c, h, wd, dtype=F32)
    w = rnd(rng, k, c, r, r, dtype=F32, scale=(2.0 / (c * r * r)) ** 0.5)
    dy = rnd(rng, n, k, 1 + (h + 2 * pad - r) // stride, 1 + (wd + 2 * pad - r) // stride, dtype=F32)
    return x, w, dy


def both(shape, x, w, dy):
    """Forward and backward data from packed filters: out of buffers that hold NaN, then added to themselves."""
    xd, wd, dyd = dev(x, F32), dev(w, F32), dev(dy, F32)
    torch.cuda.synchronize()  # (the calls below go to the default stream)
    for kind in (K.CONV_FWD, K.CONV_BWD_DATA):
        out = dev(np.full(dy.shape if kind == K.CONV_FWD else x.shape, np.nan, np.float32), F32)
        px, py = (xd, out) if kind == K.CONV_FWD else (out, dyd)
        px, pw, py = (t.data_ptr() for t in (px, wd, py))
        vx, vw, vy = (C.byref(v) for v in views(shape, px, pw, py))
        p, L = C.byref(K.ConvParams(shape[7], shape[6], 1, 1)), K.lib()
        n = L.saga_hip_conv2d_pack_bytes(kind, vx, vw, vy, p)
        packed = None
        if n:
            packed = torch.full((n // 4,), np.nan, device="cuda")
            jobs, blocks = (K.FilterPackJob * 16)(), 0
            count = L.saga_hip_conv2d_pack_jobs(kind, vx, vw, vy, p, K.ptr(packed), jobs)
            for j in jobs[:count]:
                j.first_block, blocks = blocks, blocks + j.blocks
            table = torch.frombuffer(bytearray(C.string_at(jobs, C.sizeof(K.FilterPackJob) * count)), dtype=torch.uint8).cuda()
            torch.cuda.synchronize()
            K.check(L.saga_hip_filter_pack_batched(K.ptr(table), count, blocks, None))
            run(kind, shape, px, pw, py, packed.data_ptr())
        else:
            K.conv2d(kind, xd if kind == K.CONV_FWD else dyd, wd, out, shape[7], shape[6])
        torch.cuda.synchronize()
        first = host(out).copy()
        if n:
            run(kind, shape, px, pw, py, packed.data_ptr(), 1.0)
        torch.cuda.synchronize()
        yield kind, first, host(out) if n else 2 * first


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES)
def test_against_64_bits(shape):
    x, w, dy = operands(shape)
    want = reference(shape, x, w, dy)
    for kind, got, twice in both(shape, x, w, dy):
        ref, red = want[kind], shape[1] if kind == K.CONV_FWD else shape[4]
        # six products per sixteen reduction indices, each rounding the sum by at most half a last place, at random
        bound = 2.0 ** -24 * (6 * max(red, 16) * shape[5] ** 2 / 16) ** 0.5 + 2.0 ** -24
        for a, r in ((got, ref), (twice, 2 * ref)):
            assert np.linalg.norm(a.astype(np.float64) - r) <= 2 * bound * np.linalg.norm(r)


@pytest.mark.gpu
@pytest.mark.parametrize("scales", [(-120, 80), (80, -120), (-140, 100), (-20, -100)], ids=str)
@pytest.mark.parametrize("shape", [*SHAPES, CLASSES, FEW], ids=str)
def test_small_numbers(shape, scales):
    """Operands whose low bits a bf16 cannot hold, subnormal ones among them, are multiplied with all their bits."""
    n, c, h, wd, k, r, stride, pad = shape
    x, w, dy = operands(shape)
    x, dy = (np.ldexp(a, scales[0]) for a in (x, dy))
    w = np.ldexp(w, scales[1])
    want = reference(shape, x, w, dy)
    for kind, got, _ in both(shape, x, w, dy):
        ref, red = want[kind], c if kind == K.CONV_FWD else k
        bound = 2.0 ** -24 * (6 * max(red, 16) * r ** 2 / 16) ** 0.5 + 2.0 ** -24  # (as above)
        assert np.linalg.norm(got.astype(np.float64) - ref) <= 2 * bound * np.linalg.norm(ref)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [*SHAPES, CLASSES, FEW, (1, 24, 150, 161, 24, 3, 1, 1)])
def test_numbers_without_three_parts(shape):
    """Infinities, NaNs and numbers next to the largest in either operand: where they belong, nowhere else; and what shares a
    wavefront with them is multiplied with all bits of its weights."""
    n, c, h, wd, k, r, stride, pad = shape
    x, w, dy = operands(shape)
    rng = np.random.default_rng(1)
    for value in (np.inf, -np.inf, np.nan, 3.4e38):
        for a in (x, dy):
            a.reshape(-1)[rng.integers(a.size)] = value
    w.reshape(-1)[rng.integers(w.size)] = 1.2345678e32
    if r == 1:  # (the zeros around an image times an infinity are NaN, here and in every kernel that multiplies them)
        w[rng.integers(k), rng.integers(c)] = np.inf
    want = reference(shape, x, w, dy)
    spread = reference(shape, *(a.astype(np.float64) ** 2 for a in (x, w, dy)))
    for kind, got, _ in both(shape, x, w, dy):
        with np.errstate(over="ignore"):
            ref = want[kind].astype(np.float32)
        np.testing.assert_array_equal(np.isnan(got), np.isnan(ref))
        np.testing.assert_array_equal(got[np.isinf(ref)], ref[np.isinf(ref)])
        ok = np.isfinite(ref)
        # The largest of some 10^6 errors, each a chain of `red` roundings of up to half a unit at random: 2**-24 / sqrt(3) of a partial
        # sum each, which grows like the root of its length to the sum's deviation, or to the sum itself where that is larger.
        # (Weights without their third part: some 2e-6 of a deviation on average.)
        red = (c if kind == K.CONV_FWD else k) * r * r
        size = np.sqrt(spread[kind][ok]) + np.abs(want[kind][ok])
        assert (np.abs(got[ok] - want[kind][ok]) <= 6 * (2.0 ** -24 / 3 ** 0.5 * (red / 2) ** 0.5 + 2.0 ** -24) * size).all()
