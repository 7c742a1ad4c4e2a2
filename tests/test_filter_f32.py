"""The backward filter of fp32 3x3 convolutions from split operands in LDS (csrc/filter_f32.hip): which calls go there, held on the
stub runtime; on the GPU against 64 bits, on whole numbers, whose sums are exact in 32 bits, and with operands that have no
three bf16 parts."""
import ctypes as C

import pytest
import torch

from saga_amd import kernels as K
from tests import stub_gpu
from tests.stub_gpu import on_stub

# N, C, H, W, K: whether a block has three tiles or more, and not too much in them that counts for nothing
ROUTES = {
    (600, 64, 8, 8, 64): True,
    (512, 64, 8, 8, 64): False,
    (600, 64, 8, 7, 64): False,     # narrower than a tile
    (600, 60, 8, 8, 64): False,     # channels that come in no eights
    (9, 512, 8, 8, 512): True,      # four shares of nine tiles
    (5, 136, 29, 17, 200): True,    # tiles overlap both ways; channels in part of a block
    (70, 24, 33, 29, 40): True,
    (225, 16, 9, 9, 128): False,    # four tiles to an image of little more than one
    (76, 64, 11, 11, 120): False,
    (78, 8, 12, 12, 416): False,    # an eighth of a block's input channels
}
SHAPES = [s for s, taken in ROUTES.items() if taken]
P = K.ConvParams(1, 1, 1, 1)


def view(t, address=None):
    v = K.TensorView()
    v.ptr, v.dtype = t.data_ptr() if address is None else address, K.FLOAT
    v.dims[:], v.strides[:] = list(t.shape), list(t.stride())
    return v


@on_stub
def test_routes():
    L, p = K.lib(), C.byref(P)
    for (n, c, h, w, k), taken in ROUTES.items():
        x, y, f = (view(torch.empty(d, device="meta"), a) for d, a in (((n, c, h, w), 1 << 20), ((n, k, h, w), 1 << 31), ((k, c, 3, 3), 1 << 32)))
        need = L.saga_hip_conv2d_workspace_size(K.CONV_BWD_FILTER, C.byref(x), C.byref(f), C.byref(y), p)
        one = 4 * k * c * 9
        for room in (need, one, one - 4):  # partial results enough, one (others share the pixels better, but may need a table), not even that
            stub_gpu.launched()
            rc = L.saga_hip_conv2d_bwd_filter(C.byref(x), C.byref(y), C.byref(f), p, 1.0, 0.0, 1 << 33, room, None)
            ran = [(name, blocks) for name, _, blocks, _ in stub_gpu.launched() if name == "conv_f32_bwd_filter_windows"]
            if not taken:  # (with room for one partial result and no table, whatever can run does)
                assert ran == [] or room == one, (n, c, h, w, k)
            elif room < one:
                assert rc != 0 and ran == []
            else:
                pairs = -(-k // 64) * -(-c // 64)
                assert rc == 0 and [blocks for _, blocks in ran] == ([256 // pairs * pairs] if room == need else [pairs] if c % 32 else []), (n, c, h, w, k, room)


def gradient(x, dy, f, alpha=1.0, beta=0.0):
    L, p = K.lib(), C.byref(P)
    vx, vy, vf = (C.byref(view(t)) for t in (x, dy, f))
    ws = torch.empty(L.saga_hip_conv2d_workspace_size(K.CONV_BWD_FILTER, vx, vf, vy, p), dtype=torch.uint8, device=x.device)
    K.check(L.saga_hip_conv2d_bwd_filter(vx, vy, vf, p, alpha, beta, K.ptr(ws), ws.numel(), K.stream_ptr()))


def oracle(x, dy):
    n, c, h, w = x.shape
    xp = torch.nn.functional.pad(x.double(), (1, 1, 1, 1))
    rows = lambda t: t.permute(0, 2, 3, 1).reshape(-1, t.shape[1])
    d = rows(dy.double()).t().contiguous()
    return torch.stack([torch.stack([d @ rows(xp[:, :, r:r + h, s:s + w]) for s in range(3)], -1) for r in range(3)], -2)


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["dense", "channels last", "inside"])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_exact(shape, layout):
    """Whole numbers of up to 11 bits, two parts each; sums stay below 2**24."""
    n, c, h, w, k = shape
    g = torch.Generator("cuda").manual_seed(c + h)

    def whole(ch, top):
        room = (n, ch + 3, h + 2, w + 5) if layout == "inside" else (n, ch, h, w)
        t = torch.randint(-top, top + 1, room, device="cuda", generator=g).float()
        t = t.contiguous(memory_format=torch.channels_last) if layout == "channels last" else t
        return t[:, 2:2 + ch, 1:1 + h, 3:3 + w] if layout == "inside" else t

    x, dy = whole(c, 1023), whole(k, 2)
    dy *= torch.rand(dy.shape, device="cuda", generator=g) < 0.25  # (at most n * h * w / 4 * 2046, on average far less)
    f = torch.randint(-9, 10, (k, c, 3, 3), device="cuda", generator=g).float()
    want = 2 * oracle(x, dy) + f.double()
    assert want.abs().max() < 2 ** 23
    gradient(x, dy, f, 2.0, 1.0)
    assert torch.equal(f.double(), want)


@pytest.mark.gpu
def test_no_worse_than_fp32():
    """Random operands: every product is in error by less than 2**-23 of itself (split_f32.hpp), and 32-bit sums of chains as long as a
    block's (at most 24 * 64 pixels here, times two sums, plus 32 partials) add half a unit each in the worst case."""
    n, c, h, w, k = 5, 136, 29, 17, 200
    g = torch.Generator("cuda").manual_seed(7)
    x, dy = torch.randn(n, c, h, w, device="cuda", generator=g), torch.randn(n, k, h, w, device="cuda", generator=g)
    f = torch.zeros(k, c, 3, 3, device="cuda")
    gradient(x, dy, f)
    error = (f.double() - oracle(x, dy)).abs()
    assert (error <= oracle(x.abs(), dy.abs()) * 2.0 ** -24 * (2 + 2 * 24 * 4 + 32)).all()
    assert error.norm() / oracle(x, dy).norm() < 3e-7  # (fp32 instructions: 2e-7 to 4e-7 at this size)


@pytest.mark.gpu
@pytest.mark.parametrize("scales", [(-120, 80), (80, -120), (-140, 100), (-20, -100)], ids=str)
def test_small_numbers(scales):
    """Operands whose low bits a bf16 cannot hold, subnormal ones among them: the same bound."""
    n, c, h, w, k = 70, 24, 33, 29, 40
    g = torch.Generator().manual_seed(7)  # (on the host: what makes subnormal numbers on the device is not asked here)
    x, dy = (torch.ldexp(torch.randn(n, ch, h, w, generator=g), torch.tensor(s)).cuda() for ch, s in ((c, scales[0]), (k, scales[1])))
    f = torch.zeros(k, c, 3, 3, device="cuda")
    gradient(x, dy, f)
    error, want = (f.double() - oracle(x, dy)).abs(), oracle(x, dy)
    assert error.norm() / want.norm() < 3e-7
    assert (want.abs() > 0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("value", [float("inf"), float("nan"), 3.4e38], ids=str)
def test_without_three_parts(value):
    """Such an operand reaches the sums that have it and no other."""
    n, c, h, w, k = 5, 136, 29, 17, 200
    g = torch.Generator("cuda").manual_seed(3)
    x, dy = (torch.randint(1, 4, (n, ch, h, w), device="cuda", generator=g).float() for ch in (c, k))
    x[0, 3, 5, w - 1] = x[1, 70, h - 1, 2] = value
    if value == 3.4e38:
        dy *= 0.25  # (finite products)
    f = torch.zeros(k, c, 3, 3, device="cuda")
    want = oracle(x, dy)
    gradient(x, dy, f)
    ok = torch.isfinite(want)
    assert torch.equal(torch.isfinite(f), ok)
    big = want.abs() > 1e30
    assert torch.equal(f[ok & ~big].double(), want[ok & ~big])
    assert torch.allclose(f[ok & big].double(), want[ok & big], rtol=1e-6)


# N, C, H, W, K of layers with 32 channels or fewer of a kind, whose wavefronts share a tile's rows: one block and a part of one, the lowest
# images, tiles that overlap by most of a tile, blocks with unequal numbers of tiles; and what stays with the others
FEW = {
    (130, 16, 16, 8, 16): None,     # too little work
    (420, 16, 17, 9, 8): 256,       # 16 channels of 32 are loaded
    (48, 16, 32, 32, 16): 128,
    (90, 32, 33, 17, 24): 256,
    (130, 24, 16, 31, 32): 173,
    (500, 32, 8, 9, 32): 256,       # images lower than 16 rows: blocks of 64 input channels
    (60, 72, 31, 30, 24): 256,      # 32 output channels to a block, two blocks of input channels
    (60, 24, 15, 40, 200): 256,     # the other way round
}


def _few_routes():
    L, p = K.lib(), C.byref(P)
    for (n, c, h, w, k), blocks in FEW.items():
        x, y, f = (view(torch.empty(d, device="meta"), a) for d, a in (((n, c, h, w), 1 << 20), ((n, k, h, w), 1 << 31), ((k, c, 3, 3), 1 << 32)))
        need = L.saga_hip_conv2d_workspace_size(K.CONV_BWD_FILTER, C.byref(x), C.byref(f), C.byref(y), p)
        stub_gpu.launched()
        assert L.saga_hip_conv2d_bwd_filter(C.byref(x), C.byref(y), C.byref(f), p, 1.0, 0.0, 1 << 33, need, None) == 0
        yield [b for name, _, b, _ in stub_gpu.launched() if name == "conv_f32_bwd_filter_windows"], blocks


@on_stub
def test_routes_of_few_channels():
    for ran, blocks in _few_routes():
        print(ran, blocks)
        assert ran == ([] if blocks is None else [blocks])


@pytest.mark.gpu
@pytest.mark.parametrize("value", [None, float("inf"), float("nan")], ids=str)
@pytest.mark.parametrize("shape", [s for s, blocks in FEW.items() if blocks], ids=str)
def test_few_channels(shape, value):
    """Exact on whole numbers, as above; an operand without three parts reaches the sums that have it and no other."""
    n, c, h, w, k = shape
    g = torch.Generator("cuda").manual_seed(c + h)
    x = torch.randint(-1023, 1024, (n, c, h, w), device="cuda", generator=g).float()
    dy = torch.randint(-2, 3, (n, k + 3, h + 2, w + 5), device="cuda", generator=g).float()[:, 2:2 + k, 1:1 + h, 3:3 + w]
    dy *= torch.rand(dy.shape, device="cuda", generator=g) < 0.25
    f = torch.randint(-9, 10, (k, c, 3, 3), device="cuda", generator=g).float()
    if value is not None:
        x[0, c - 1, h - 1, w - 1] = x[n // 2, 3, 5, 0] = value
    want = 2 * oracle(x, dy) + f.double()
    gradient(x, dy, f, 2.0, 1.0)
    ok = torch.isfinite(want)
    assert torch.equal(torch.isfinite(f), ok) and want[ok].abs().max() < 2 ** 23
    assert torch.equal(f[ok].double(), want[ok])
