"""fp16 3x3 convolutions from windows in LDS (csrc/window_f16.hip): which calls go there and in what form, held on the stub runtime;
on the GPU against 64 bits, on small whole numbers: every sum is exact in 32 bits and every result in 16."""
import ctypes as C

import pytest
import torch

from saga_amd import kernels as K
from tests import stub_gpu
from tests.stub_gpu import on_stub

# N, C, H, W, K: the forward launch's tile rows, columns in 32s of a wavefront, wavefronts along the pixels, rounds of loads, patches
SHAPES = {
    (262, 72, 14, 14, 256): (4, 2, 2, 6, 0),   # windows over several images; a half slice at the end
    (58, 40, 30, 30, 200): (4, 2, 2, 8, 0),    # channels in part of a block
    (6, 24, 95, 98, 256): (4, 2, 2, 10, 0),    # the filter as it is
    (3, 40, 130, 140, 256): (4, 2, 2, 7, 1),   # patches in part outside, right and below
    (250, 72, 28, 29, 40): (4, 2, 4, 8, 0),
    (14, 72, 120, 121, 56): (4, 2, 4, 10, 0),
    (4, 72, 224, 230, 64): (4, 2, 4, 8, 1),
    (8, 48, 70, 71, 48): (2, 2, 4, 8, 0),
    (3, 64, 113, 114, 96): (2, 2, 4, 10, 0),
    (2, 40, 130, 150, 80): (2, 2, 4, 7, 1),
    (40, 16, 20, 21, 24): (2, 1, 4, 5, 0),
    (4, 8, 100, 90, 16): (2, 1, 4, 8, 0),
    (2, 16, 60, 220, 8): (2, 1, 4, 4, 1),
    (8, 21, 70, 71, 70): (2, 2, 4, 8, 0),      # channel counts that go through padded copies
}
P = K.ConvParams(1, 1, 1, 1)


def view(t, address=None):
    v = K.TensorView()
    v.ptr, v.dtype = t.data_ptr() if address is None else address, K.HALF
    v.dims[:], v.strides[:] = list(t.shape), list(t.stride())
    return v


@on_stub
def test_forms():
    L, p = K.lib(), C.byref(P)
    cl = lambda *d: torch.empty(d, dtype=torch.float16, device="meta").contiguous(memory_format=torch.channels_last)

    def forward(n, c, h, w, k, room=None, stats=False):
        x, f, y = view(cl(n, c, h, w), 1 << 20), view(cl(k, c, 3, 3), 1 << 31), view(cl(n, k, h, w), 1 << 30)
        a = C.byref(x), C.byref(f), C.byref(y)
        room = L.saga_hip_conv2d_workspace_size(K.CONV_FWD, *a, p) if room is None else room
        stub_gpu.launched()
        if stats:
            rows = C.c_int(0)
            floats = L.saga_hip_conv2d_fwd_bnstats_size(*a, p)
            assert L.saga_hip_conv2d_fwd_bnstats(*a, p, 1.0, 1 << 32, room, 1 << 33, floats, C.byref(rows), None) == 0
            assert 0 < rows.value * k * 8 <= floats
        else:
            assert L.saga_hip_conv2d_fwd(*a, p, 1.0, 0.0, 1 << 32, room, None) == 0
        return [t[:3] + (t[5], t[7]) for name, t, *_ in stub_gpu.launched() if name == "conv_window"]

    for shape, form in SHAPES.items():
        assert forward(*shape) == [form], shape
        # training: from 2**17 values of a channel on, or with one slice of channels (half and wide forms: of 32, the others: of 16)
        n, c, h, w, k = shape
        slice = 32 if form[:3] in ((4, 2, 2), (2, 2, 4)) else 16
        assert forward(*shape, stats=True) == ([form] if n * h * w >= 1 << 17 or c <= slice else []), shape
    for n, h, taken in ((167, 28, 0), (168, 28, 1), (255, 28, 1), (256, 28, 1), (31, 65, 0), (32, 65, 1)):  # 130928, 131712 ... values
        assert len(forward(n, 128, h, h, 128, stats=True)) == taken, (n, h)
    assert forward(262, 72, 14, 14, 256, room=0) == []  # no room for the packed filter, and nobody has it
    assert forward(6, 24, 95, 98, 256, room=0) == [(4, 2, 2, 10, 0)]
    assert forward(4, 72, 14, 14, 256) == []  # a small grid
    assert forward(106, 128, 17, 17, 16) == [] and len(forward(174, 392, 14, 14, 16)) == 1  # few results of a filter to pack
    assert forward(200, 16, 3, 330, 40) == []  # a row too long for a window, patches of which the image fills little


def rows(t):
    return t.permute(0, 2, 3, 1).reshape(-1, t.shape[1])


def oracle(x, w):
    n, _, h, wd = x.shape
    xp, wt = torch.nn.functional.pad(x.double(), (1, 1, 1, 1)), w.double()
    y = sum(rows(xp[:, :, r:r + h, s:s + wd]) @ wt[:, :, r, s].t().contiguous() for r in range(3) for s in range(3))
    return y.reshape(n, h, wd, -1).permute(0, 3, 1, 2)


def whole(g, *shape, top=2, wide=0):
    """Small whole numbers, channels-last; wide: a slice of a tensor with more channels."""
    n, c, h, w = shape
    t = torch.randint(-top, top + 1, (n, c + wide, h, w), device="cuda", generator=g).half().contiguous(memory_format=torch.channels_last)
    return t[:, wide // 2:wide // 2 + c]


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_forward(shape):
    n, c, h, w, k = shape
    g = torch.Generator("cuda").manual_seed(c + w)
    L, p, st = K.lib(), C.byref(P), K.stream_ptr()
    x, f, y = whole(g, n, c, h, w, wide=16), whole(g, k, c, 3, 3), whole(g, n, k, h, w, wide=16)
    a = [C.byref(view(t)) for t in (x, f, y)]
    ws = torch.empty(L.saga_hip_conv2d_workspace_size(K.CONV_FWD, *a, p), dtype=torch.uint8, device="cuda")
    want, old = oracle(x, f), y.double()
    K.check(L.saga_hip_conv2d_fwd(*a, p, 0.5, 1.0, K.ptr(ws), ws.numel(), st))
    assert torch.equal(y, (0.5 * want + old).half())
    floats = L.saga_hip_conv2d_fwd_bnstats_size(*a, p)
    part, count = torch.full((floats // 4,), float("nan"), device="cuda"), C.c_int(0)
    K.check(L.saga_hip_conv2d_fwd_bnstats(*a, p, 1.0, K.ptr(ws), ws.numel(), K.ptr(part), floats, C.byref(count), st))
    assert torch.equal(y, want.half())
    sums = part[: count.value * k * 2].reshape(-1, k, 2).double().sum(0)
    assert torch.equal(sums, torch.stack([want.sum((0, 2, 3)), (want ** 2).sum((0, 2, 3))], 1))
    # a folded norm (scale 2, shift b - 2m), a residual and relu
    z, b, m = whole(g, n, k, h, w), *(torch.randint(-3, 4, (k,), device="cuda", generator=g).float() for _ in range(2))
    two, one = torch.full_like(b, 2.0), torch.ones_like(b)
    K.check(L.saga_hip_conv2d_fwd_bn_infer(*a, C.byref(view(z)), p, K.ptr(two), K.ptr(b), K.ptr(m), K.ptr(one), 0.0, K.BN_RELU | K.BN_ADD,
                                           K.ptr(ws), ws.numel(), st))
    per = lambda t: t.double().reshape(1, -1, 1, 1)
    folded = (2 * (want - per(m)) + per(b) + z.double()).clamp(min=0).half()
    assert torch.equal(y, folded)
    # the same from a filter packed beforehand, as an inference program has it
    n = L.saga_hip_conv2d_pack_bytes(K.CONV_FWD, *a, p)
    assert (n > 0) == (c > 32)
    if n:
        packed, job = torch.empty(n, dtype=torch.uint8, device="cuda"), (K.FilterPackJob * 16)()
        assert L.saga_hip_conv2d_pack_jobs(K.CONV_FWD, *a, p, K.ptr(packed), job) == 1
        table = torch.frombuffer(bytearray(job)[:C.sizeof(K.FilterPackJob)], dtype=torch.uint8).cuda()
        K.check(L.saga_hip_filter_pack_batched(K.ptr(table), 1, job[0].blocks, st))
        y.zero_()
        e = K.ConvExtras(packed=K.ptr(packed), s=K.ptr(two), b=K.ptr(b), m=K.ptr(m), v=K.ptr(one), z=C.pointer(view(z)), relu=1)
        K.check(L.saga_hip_conv2d_fwd_ex(*a, p, 0.0, C.byref(e), None, 0, st))
        assert torch.equal(y, folded)



@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_backward_data(shape):
    n, k, h, w, c = shape  # the roles of the channels exchanged: the same forms
    g = torch.Generator("cuda").manual_seed(c + h)
    L, p, st = K.lib(), C.byref(P), K.stream_ptr()
    dy, f, dx = whole(g, n, k, h, w, wide=16), whole(g, k, c, 3, 3), whole(g, n, c, h, w, wide=16)
    vy, vf, vx = (C.byref(view(t)) for t in (dy, f, dx))
    ws = torch.empty(L.saga_hip_conv2d_workspace_size(K.CONV_BWD_DATA, vx, vf, vy, p), dtype=torch.uint8, device="cuda")
    want, old = oracle(dy, f.transpose(0, 1).flip(2, 3)), dx.double()
    wt = f.permute(1, 2, 3, 0).contiguous() if k % 8 == 0 else None
    K.check(L.saga_hip_conv2d_bwd_data_wt(vy, vf, K.ptr(wt) if wt is not None else None, vx, p, 1.0, 1.0, K.ptr(ws), ws.numel(), st))
    assert torch.equal(dx, (want + old).half())
    K.check(L.saga_hip_conv2d_bwd_data(vy, vf, vx, p, 1.0, 0.0, K.ptr(ws), ws.numel(), st))
    assert torch.equal(dx, want.half())
    nbytes = L.saga_hip_conv2d_bwd_data_bnbwd_size(vy, vf, vx, p)
    if not nbytes or wt is None:
        return
    # linked to the backward of a norm (mean 1, scale 1, shift 0) and a relu
    xn, one, zero = whole(g, n, c, h, w, top=3), torch.ones(c, device="cuda"), torch.zeros(c, device="cuda")
    part = torch.full((nbytes // 4,), float("nan"), device="cuda")
    link = K.BnBwdLink(C.pointer(view(xn)), K.ptr(one), K.ptr(zero), K.ptr(one), K.ptr(one), K.BN_RELU, 0, K.ptr(part), nbytes)
    K.check(L.saga_hip_conv2d_bwd_data_bnbwd(vy, vf, K.ptr(wt), vx, p, 1.0, 0.0, K.ptr(ws), ws.numel(), C.byref(link), st))
    masked = torch.where(xn.double() - 1 > 0, want, torch.zeros_like(want))
    assert torch.equal(dx.double(), masked)
    sums = part[: link.partial_rows * c * 2].reshape(-1, c, 2).double().sum(0)
    assert torch.equal(sums, torch.stack([masked.sum((0, 2, 3)), (masked * (xn.double() - 1)).sum((0, 2, 3))], 1))
