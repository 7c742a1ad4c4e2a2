"""The backward filter of fp16 3x3 convolutions over image strips in LDS (csrc/filter_strips.hip): which calls go there, held on
the stub runtime; on the GPU against 64 bits, on small whole numbers, whose sums are exact in 32 bits."""
import ctypes as C

import pytest
import torch

from saga_amd import kernels as K
from tests import stub_gpu
from tests.stub_gpu import on_stub

# N, C, H, W, K: whether a block has three tiles or more, and not too much of them twice
ROUTES = {
    (57, 192, 16, 16, 192): True,    # 28 shares of 57 tiles
    (56, 192, 16, 16, 192): False,
    (57, 192, 16, 15, 192): False,   # narrower than a tile of 16 rows, shorter than one of 8 columns
    (60, 192, 16, 7, 192): False,
    (30, 200, 32, 11, 136): True,    # 8 columns x 32 rows, channels in part of a block
    (120, 126, 28, 23, 126): True,   # 8 x 28; channel counts and tensors that go through padded copies
    (45, 192, 23, 31, 192): True,    # 16 x 14; tiles overlap both ways
    (64, 128, 40, 39, 128): True,    # an overlap of half a tile both ways
    (23, 192, 29, 31, 192): True,    # 16 x 16
    (15, 192, 23, 19, 192): False,   # too much of a tile is in others too
    (9, 512, 17, 33, 512): False,
    (70, 70, 28, 9, 70): False,
    (11, 16, 67, 67, 368): False,    # a block of channels of which most are not there
}
SHAPES = [s for s, strips in ROUTES.items() if strips]


def view(t, address=None):
    v = K.TensorView()
    v.ptr, v.dtype = t.data_ptr() if address is None else address, K.HALF
    v.dims[:], v.strides[:] = list(t.shape), list(t.stride())
    return v


@pytest.mark.parametrize("shape", ROUTES, ids=str)
@on_stub
def test_route(shape):
    n, c, h, w, k = shape
    L, p = K.lib(), C.byref(K.ConvParams(1, 1, 1, 1))
    cl = lambda *d: torch.empty(d, dtype=torch.float16, device="meta").contiguous(memory_format=torch.channels_last)
    x, y, f = view(cl(n, c, h, w), 1 << 20), view(cl(n, k, h, w), 1 << 30), view(cl(k, c, 3, 3), 1 << 31)
    need = L.saga_hip_conv2d_workspace_size(K.CONV_BWD_FILTER, C.byref(x), C.byref(f), C.byref(y), p)
    before = stub_gpu.launches("conv_bwd_filter_strips"), stub_gpu.launches("conv_bwd_filter_dma")
    assert L.saga_hip_conv2d_bwd_filter(C.byref(x), C.byref(y), C.byref(f), p, 1.0, 0.0, 1 << 32, need, None) == 0
    ran = stub_gpu.launches("conv_bwd_filter_strips") - before[0], stub_gpu.launches("conv_bwd_filter_dma") - before[1]
    assert ran == ((1, 0) if ROUTES[tuple(shape)] else (0, 1))


def gradient(x, dy, f, beta):
    L, p = K.lib(), C.byref(K.ConvParams(1, 1, 1, 1))
    vx, vy, vf = (C.byref(view(t)) for t in (x, dy, f))
    ws = torch.empty(L.saga_hip_conv2d_workspace_size(K.CONV_BWD_FILTER, vx, vf, vy, p), dtype=torch.uint8, device=x.device)
    K.check(L.saga_hip_conv2d_bwd_filter(vx, vy, vf, p, 1.0, beta, K.ptr(ws), ws.numel(), K.stream_ptr()))


def oracle(x, dy):
    n, c, h, w = x.shape
    xp = torch.nn.functional.pad(x.double(), (1, 1, 1, 1))
    rows = lambda t: t.permute(0, 2, 3, 1).reshape(-1, t.shape[1])
    d = rows(dy.double()).t().contiguous()
    return torch.stack([torch.stack([d @ rows(xp[:, :, r:r + h, s:s + w]) for s in range(3)], -1) for r in range(3)], -2)


@pytest.mark.gpu
@pytest.mark.parametrize("wide,beta", [(0, 0.0), (24, 1.0)])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_exact(shape, wide, beta):
    """Dense tensors, and slices of tensors with more channels; the sums are whole numbers far below 2**24, rounded once."""
    n, c, h, w, k = shape
    g = torch.Generator("cuda").manual_seed(c + h)

    def whole(m, ch, hh, ww):
        t = torch.randint(-2, 3, (m, ch + wide, hh, ww), device="cuda", generator=g).half().contiguous(memory_format=torch.channels_last)
        return t[:, wide // 2 // 8 * 8:][:, :ch]

    x, dy = whole(n, c, h, w), whole(n, k, h, w)
    f = torch.randint(-9, 10, (k, c, 3, 3), device="cuda", generator=g).half().contiguous(memory_format=torch.channels_last)
    want = (oracle(x, dy) + beta * f.double()).half()
    gradient(x, dy, f, beta)
    assert torch.equal(f, want)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(23, 192, 29, 31, 192), (30, 200, 32, 11, 136)], ids=str)
def test_infinities(shape):
    """An infinity at a border reaches the taps that see it and no other: pixels outside the image have no products."""
    n, c, h, w, k = shape
    g = torch.Generator("cuda").manual_seed(1)
    half = lambda *d: torch.randint(1, 3, d, device="cuda", generator=g).half().contiguous(memory_format=torch.channels_last)
    x, dy = half(n, c, h, w), half(n, k, h, w)
    x[0, 3, 5, w - 1] = x[1, 70, h - 1, 2] = x[2, 130, 0, 0] = float("inf")
    f = torch.zeros(k, c, 3, 3, device="cuda", dtype=torch.float16).contiguous(memory_format=torch.channels_last)
    want = oracle(x, dy)
    gradient(x, dy, f, 0.0)
    assert torch.equal(torch.isfinite(f), torch.isfinite(want)) and not torch.isfinite(want).all()
    ok = torch.isfinite(want)
    assert torch.equal(f[ok], want[ok].half())


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_infinities_where_tiles_overlap(shape):
    """They meet the zeros of pixels seen before under no tap: sums that should be infinite are, all others are as they should be."""
    n, c, h, w, k = shape
    g = torch.Generator("cuda").manual_seed(2)
    half = lambda *d: (torch.randint(1, 3, d, device="cuda", generator=g) / 8).half().contiguous(memory_format=torch.channels_last)
    x, dy = half(n, c, h, w), half(n, k, h, w)
    x[0, 3, h // 2, w // 2], x[1, c - 1, h - 15, w - 7] = float("inf"), float("-inf")
    x[2, 5, h - 14, :], x[3, 40, :, w - 8] = float("inf"), float("inf")
    x[4, 17, h // 2, w // 2] = float("nan")
    f = torch.zeros(k, c, 3, 3, device="cuda", dtype=torch.float16).contiguous(memory_format=torch.channels_last)
    want = oracle(x, dy).half()
    gradient(x, dy, f, 0.0)
    assert torch.equal(torch.isnan(f), torch.isnan(want)) and torch.isinf(want).any()
    ok = ~torch.isnan(want)
    assert torch.equal(f[ok], want[ok])
