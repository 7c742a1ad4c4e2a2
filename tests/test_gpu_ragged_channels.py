"""fp16 convolutions whose output rows lie off the grid of 16 bytes or end inside it: odd numbers of channels, odd pitches and
addresses, through every kernel that writes such rows - against 64 bits, on small whole numbers: every sum is exact in 32
bits and every result in 16 - and nothing beside the rows is touched."""
import ctypes as C

import pytest
import torch

from saga_amd import kernels as K
from tests import stub_gpu
from tests.stub_gpu import on_stub

HALF = torch.float16
# N, C, H, W, K, filter, stride, channels beside the output's in a row, halves in front of it: the forward launch
SHAPES = {
    (37, 48, 25, 25, 398, 1, 1, 0, 0): "conv_gather_gemm_dma",
    (40, 32, 24, 30, 263, 1, 1, 3, 1): "conv_gather_gemm_dma",
    (60, 40, 30, 31, 61, 1, 1, 0, 1): "conv_gather_gemm_dma",       # 64 channels to a tile
    (140, 48, 28, 29, 130, 3, 2, 1, 0): "conv_gather_gemm_dma",     # backward: residue classes
    (60, 16, 29, 29, 181, 3, 1, 0, 0): "conv_window",
    (3, 40, 130, 140, 250, 3, 1, 5, 1): "conv_window",              # patches
    (40, 16, 20, 21, 21, 3, 1, 0, 1): "conv_window",                # 32 channels to a block
    (2, 24, 11, 13, 33, 3, 1, 2, 1): "stream_f16_k",
    (1, 64, 14, 14, 131, 1, 1, 0, 0): "stream_f16_k",
    (9, 16, 19, 17, 66, 5, 1, 0, 1): "stream_f16_k",
    (2, 13, 12, 12, 7, 3, 2, 0, 0): "stream_f16_k",                 # operands through padded copies
    (33, 21, 40, 41, 150, 3, 1, 0, 1): "conv_window",
}


def out_size(shape):
    n, c, h, w, k, r, stride, _, _ = shape
    return (h + 2 * (r // 2) - r) // stride + 1, (w + 2 * (r // 2) - r) // stride + 1


@on_stub
def test_the_kernels_they_are_for():
    L = K.lib()
    for shape, kernel in SHAPES.items():
        n, c, h, w, k, r, stride, wide, shift = shape
        x, f = (torch.empty(d, dtype=HALF, device="meta").contiguous(memory_format=torch.channels_last) for d in ((n, c, h, w), (k, c, r, r)))
        y = torch.empty(n, k + wide, *out_size(shape), dtype=HALF, device="meta").contiguous(memory_format=torch.channels_last)[:, :k]
        views = [K.TensorView() for _ in range(3)]
        for v, t, at in zip(views, (x, f, y), (1 << 20, 1 << 31, (1 << 30) + 2 * shift)):
            v.ptr, v.dtype = at, K.HALF
            v.dims[:], v.strides[:] = list(t.shape), list(t.stride())
        a, p = [C.byref(v) for v in views], C.byref(K.ConvParams(r // 2, stride, 1, 1))
        room = L.saga_hip_conv2d_workspace_size(K.CONV_FWD, *a, p)
        stub_gpu.launched()
        assert L.saga_hip_conv2d_fwd(*a, p, 1.0, 0.0, 1 << 32, room, None) == 0
        assert stub_gpu.launched()[-1][0] == kernel, shape


def slice_of(n, c, h, w, wide, shift):
    """A slice of a tensor of more channels, some halves behind an aligned address; and all of that memory."""
    flat = torch.full((n * h * w * (c + wide) + shift,), -9.0, dtype=HALF, device="cuda")
    return flat[shift:].view(n, h, w, c + wide)[..., :c].permute(0, 3, 1, 2), flat


def whole(g, *shape, top=2):
    return torch.randint(-top, top + 1, shape, device="cuda", generator=g).half().contiguous(memory_format=torch.channels_last)


def beside(t, flat):
    """The values of the memory that are not the tensor's."""
    keep = flat.clone()
    view = keep[flat.numel() - t.shape[0] * t.shape[2] * t.shape[3] * t.stride(3):].view(t.shape[0], t.shape[2], t.shape[3], t.stride(3))
    view[..., :t.shape[1]] = -9.0
    return keep


def conv64(x, w, stride):
    n, c, h, wd = x.shape
    r = w.shape[2]
    p, q = (h + 2 * (r // 2) - r) // stride + 1, (wd + 2 * (r // 2) - r) // stride + 1
    xp, wt = torch.nn.functional.pad(x.double(), (r // 2,) * 4), w.double()
    y = sum(xp[:, :, a:a + stride * (p - 1) + 1:stride, b:b + stride * (q - 1) + 1:stride].permute(0, 2, 3, 1).reshape(-1, c)
            @ wt[:, :, a, b].t().contiguous() for a in range(r) for b in range(r))
    return y.view(n, p, q, -1).permute(0, 3, 1, 2)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_forward(shape):
    n, c, h, w, k, r, stride, wide, shift = shape
    g = torch.Generator("cuda").manual_seed(k)
    L, p, st = K.lib(), C.byref(K.ConvParams(r // 2, stride, 1, 1)), K.stream_ptr()
    x, f = whole(g, n, c, h, w), whole(g, k, c, r, r, top=1)
    want = conv64(x, f, stride)
    (y, mem), (z, _) = (slice_of(n, k, *out_size(shape), wide, shift) for _ in range(2))
    z.copy_(whole(g, *z.shape))
    y.copy_(z)
    v = lambda t: C.byref(K.view(t))
    ws = torch.empty(max(16, L.saga_hip_conv2d_workspace_size(K.CONV_FWD, v(x), v(f), v(y), p)), dtype=torch.uint8, device="cuda")
    K.check(L.saga_hip_conv2d_fwd(v(x), v(f), v(y), p, 0.5, 1.0, K.ptr(ws), ws.numel(), st))
    assert torch.equal(y, (0.5 * want + z.double()).half())
    K.check(L.saga_hip_conv2d_fwd(v(x), v(f), v(y), p, 1.0, 0.0, K.ptr(ws), ws.numel(), st))
    assert torch.equal(y, want.half())
    # a folded norm (scale 2, shift b - 2m), a residual and relu
    b, m = (torch.randint(-3, 4, (k,), device="cuda", generator=g).float() for _ in range(2))
    two, one = torch.full_like(b, 2.0), torch.ones_like(b)
    K.check(L.saga_hip_conv2d_fwd_bn_infer(v(x), v(f), v(y), v(z), p, K.ptr(two), K.ptr(b), K.ptr(m), K.ptr(one), 0.0, K.BN_RELU | K.BN_ADD,
                                           K.ptr(ws), ws.numel(), st))
    per = lambda t: t.double().view(1, -1, 1, 1)
    assert torch.equal(y, (2 * (want - per(m)) + per(b) + z.double()).clamp(min=0).half())
    assert (beside(y, mem) == -9.0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_backward(shape):
    """Gradients of layers with so many input channels (their rows are dx's), and of filters of so many."""
    n, k, h, w, c, r, stride, wide, shift = shape  # the roles exchanged
    g = torch.Generator("cuda").manual_seed(c)
    L, p, st = K.lib(), C.byref(K.ConvParams(r // 2, stride, 1, 1)), K.stream_ptr()
    ph, pw = out_size(shape)
    f, dy, x = whole(g, k, c, r, r, top=1), whole(g, n, k, ph, pw), whole(g, n, c, h, w, top=1)
    # dx by the transposed convolution in 64 bits: dy spread over the stride
    spread = torch.zeros(n, k, (ph - 1) * stride + 1, (pw - 1) * stride + 1, dtype=torch.float64, device="cuda")
    spread[:, :, ::stride, ::stride] = dy.double()
    rest = lambda full, have: full + 2 * (r // 2) - r + 1 - have  # positions that no filter begins at
    spread = torch.nn.functional.pad(spread, (r - 1, r - 1 + rest(w, spread.shape[3]), r - 1, r - 1 + rest(h, spread.shape[2])))
    wt = f.double().flip(2, 3).transpose(0, 1)
    full = sum(spread[:, :, a:spread.shape[2] - r + 1 + a, b:spread.shape[3] - r + 1 + b].permute(0, 2, 3, 1).reshape(-1, k)
               @ wt[:, :, a, b].t().contiguous() for a in range(r) for b in range(r))
    full = full.view(n, spread.shape[2] - r + 1, spread.shape[3] - r + 1, c).permute(0, 3, 1, 2)
    want = full[:, :, r // 2:r // 2 + h, r // 2:r // 2 + w]
    (dx, mem), (old, _) = (slice_of(n, c, h, w, wide, shift) for _ in range(2))
    old.copy_(whole(g, *old.shape))
    dx.copy_(old)
    v = lambda t: C.byref(K.view(t))
    ws = torch.empty(max(16, L.saga_hip_conv2d_workspace_size(K.CONV_BWD_DATA, v(dx), v(f), v(dy), p)), dtype=torch.uint8, device="cuda")
    K.check(L.saga_hip_conv2d_bwd_data(v(dy), v(f), v(dx), p, 1.0, 1.0, K.ptr(ws), ws.numel(), st))
    assert torch.equal(dx, (want + old.double()).half())
    K.check(L.saga_hip_conv2d_bwd_data(v(dy), v(f), v(dx), p, 1.0, 0.0, K.ptr(ws), ws.numel(), st))
    assert torch.equal(dx, want.half())
    assert (beside(dx, mem) == -9.0).all()
    # the filter's gradient, of a few pixels (sums that 16 bits hold): x and dy through one launch that copies both
    dy.mul_(torch.rand(dy.shape, device="cuda", generator=g) < 200.0 / (n * ph * pw))
    dw = torch.full_like(f, float("nan"))
    ws = torch.empty(max(16, L.saga_hip_conv2d_workspace_size(K.CONV_BWD_FILTER, v(x), v(dw), v(dy), p)), dtype=torch.uint8, device="cuda")
    K.check(L.saga_hip_conv2d_bwd_filter(v(x), v(dy), v(dw), p, 1.0, 0.0, K.ptr(ws), ws.numel(), st))
    xp = torch.nn.functional.pad(x.double(), (r // 2,) * 4)
    dyr = dy.double().permute(0, 2, 3, 1).reshape(-1, k).t().contiguous()
    for a in range(r):
        for b in range(r):
            xr = xp[:, :, a:a + stride * (ph - 1) + 1:stride, b:b + stride * (pw - 1) + 1:stride].permute(0, 2, 3, 1).reshape(-1, c).contiguous()
            assert torch.equal(dw[:, :, a, b], (dyr @ xr).half())
