"""The stem of an image network in one launch (csrc/stem_f16.hip): against 64 bits, on small whole numbers that every sum and every
result holds exactly; bit for bit the launches that it replaces, with what is not a number; and through the engine, whoever looks
at the tensors in between."""
import ctypes as C

import numpy as np
import pytest
import torch

from saga_amd import api as S
from saga_amd import kernels as K
from tests import stub_gpu
from tests.stub_gpu import on_stub
from tests.test_engine_plan import norm_params

HALF = torch.float16
# N, H, W, K, columns of the filter, pad, halves in front of the image
SHAPES = [(1, 224, 224, 64, 7, 3, 0), (2, 193, 193, 64, 7, 3, 0), (3, 29, 131, 64, 7, 3, 1), (1, 7, 7, 8, 7, 0, 0), (2, 9, 5, 16, 5, 3, 1),
          (1, 5, 258, 40, 7, 3, 0), (40, 65, 63, 32, 7, 2, 0), (300, 33, 40, 64, 8, 3, 0), (2, 30, 700, 64, 7, 3, 0), (3, 64, 127, 56, 6, 1, 1),
          (1, 16, 128, 64, 7, 3, 0), (1, 16, 130, 64, 7, 3, 0), (5, 300, 16, 24, 7, 3, 0)]


def dims(shape):
    n, h, w, k, s, pad, _ = shape
    p, q = (h + 2 * pad - 7) // 2 + 1, (w + 2 * pad - s) // 2 + 1
    return p, q, (p - 1) // 2 + 1, (q - 1) // 2 + 1


def channels_last(n, c, h, w, shift=0, wide=0):
    flat = torch.zeros(n * h * w * (c + wide) + shift, dtype=HALF, device="cuda")
    return flat[shift:].view(n, h, w, c + wide)[..., :c].permute(0, 3, 1, 2)


def operands(shape, wide=8):
    n, h, w, k, s, pad, shift = shape
    g = torch.Generator("cuda").manual_seed(h + w + k)
    x, f = channels_last(n, 3, h, w, shift), channels_last(k, 3, 7, s)
    x.copy_(torch.randint(-2, 3, x.shape, device="cuda", generator=g))
    f.copy_(torch.randint(-1, 2, f.shape, device="cuda", generator=g))
    b, m = (torch.randint(-3, 4, (k,), device="cuda", generator=g).float() for _ in range(2))
    two = torch.full_like(b, 2.0)
    y = channels_last(n, k, *dims(shape)[2:], wide=wide)
    return x, f, two, b, m, torch.ones_like(b), y


def fused(shape, x, f, s, b, m, v, y):
    view = lambda t: C.byref(K.view(t))
    p = K.ConvParams(shape[5], 2, 1, 1)
    assert K.lib().saga_hip_conv2d_fwd_bn_maxpool_ok(view(x), view(f), view(y), C.byref(p), 3, 1, 2)
    K.check(K.lib().saga_hip_conv2d_fwd_bn_maxpool(view(x), view(f), view(y), C.byref(p), K.ptr(s), K.ptr(b), K.ptr(m), K.ptr(v), 0.0, 3, 1, 2,
                                                   K.stream_ptr()))


def apart(shape, x, f, s, b, m, v):
    """The launches that it replaces."""
    n, h, w, k, _, pad, _ = shape
    p, q, pp, qp = dims(shape)
    L, view, cp = K.lib(), lambda t: C.byref(K.view(t)), C.byref(K.ConvParams(pad, 2, 1, 1))
    mid, y = channels_last(n, k, p, q), channels_last(n, k, pp, qp)
    ws = torch.empty(max(16, L.saga_hip_conv2d_workspace_size(K.CONV_FWD, view(x), view(f), view(mid), cp)), dtype=torch.uint8, device="cuda")
    K.check(L.saga_hip_conv2d_fwd_bn_infer(view(x), view(f), view(mid), None, cp, K.ptr(s), K.ptr(b), K.ptr(m), K.ptr(v), 0.0, K.BN_RELU,
                                           K.ptr(ws), ws.numel(), K.stream_ptr()))
    K.check(L.saga_hip_pool_fwd(K.POOL_MAX, view(mid), view(y), None, 3, 1, 2, K.stream_ptr()))
    return y


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_against_64_bits(shape):
    n, h, w, k, s, pad, _ = shape
    p, q, pp, qp = dims(shape)
    ops = operands(shape)
    x, f, two, b, m, _, y = ops
    whole = y.as_strided((n, pp, qp, k + 8), (pp * qp * (k + 8), qp * (k + 8), k + 8, 1))
    whole.fill_(-7.0)
    fused(shape, *ops)
    xp = torch.nn.functional.pad(x.double(), (pad,) * 4)
    want = sum(xp[:, :, r:r + 2 * p - 1:2, c:c + 2 * q - 1:2].permute(0, 2, 3, 1).reshape(-1, 3) @ f.double()[:, :, r, c].t().contiguous()
               for r in range(7) for c in range(s)).view(n, p, q, k).permute(0, 3, 1, 2)
    per = lambda t: t.double().view(1, -1, 1, 1)
    want = torch.nn.functional.max_pool2d((2 * (want - per(m)) + per(b)).clamp(min=0), 3, 2, 1)
    assert torch.equal(y.double(), want)
    assert (whole[..., k:] == -7.0).all()  # the channels beside it


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [SHAPES[1], SHAPES[2], SHAPES[7]], ids=str)
def test_the_same_bits_as_apart(shape):
    ops = operands(shape)
    x, f, s, b, m, v, y = ops
    g = torch.Generator("cuda").manual_seed(1)
    x.copy_(torch.randn(x.shape, device="cuda", generator=g))
    f.copy_(torch.randn(f.shape, device="cuda", generator=g) * 0.1)
    for t in (s, v):
        t.uniform_(0.5, 1.5, generator=g)
    x[0, 1, 3, 4], x[-1, 0, -2, -3] = float("nan"), 6e4
    fused(shape, *ops)
    want = apart(shape, x, f, s, b, m, v)
    assert want.isnan().any() and not want.isnan().all()
    assert torch.equal(y.isnan(), want.isnan()) and torch.equal(y.nan_to_num(-1.0), want.nan_to_num(-1.0))


def test_what_it_does_not_take():
    v = lambda *d: K.view(torch.empty(d, dtype=HALF, device="meta").contiguous(memory_format=torch.channels_last))
    def ok(x, f, y, pad=3, stride=2, pool=(3, 1, 2)):
        for t in (x, f, y):
            t.ptr = 1 << 20
        return K.lib().saga_hip_conv2d_fwd_bn_maxpool_ok(C.byref(x), C.byref(f), C.byref(y), C.byref(K.ConvParams(pad, stride, 1, 1)), *pool)
    assert ok(v(2, 3, 64, 64), v(64, 3, 7, 7), v(2, 64, 16, 16))
    assert not ok(v(2, 3, 64, 64), v(64, 3, 7, 7), v(2, 64, 16, 16), pool=(2, 0, 2))
    assert not ok(v(2, 3, 64, 64), v(64, 3, 7, 7), v(2, 64, 15, 16))
    assert not ok(v(2, 3, 64, 64), v(72, 3, 7, 7), v(2, 72, 16, 16))
    assert not ok(v(2, 4, 64, 64), v(64, 4, 7, 7), v(2, 64, 16, 16))
    assert not ok(v(2, 3, 64, 64), v(64, 3, 5, 5), v(2, 64, 16, 16), pad=2)
    assert not ok(v(2, 3, 32, 1100), v(64, 3, 7, 7), v(2, 64, 8, 275))  # rows of which no strip fits


@pytest.mark.parametrize("front", [4, 8])
@on_stub
def test_a_part_of_a_wider_tensor(front):
    """Channels behind 4 others lie at no address of whole vectors: the launches are apart, and what is between them has memory."""
    rng = np.random.default_rng(4)
    tensor = lambda *d: S.Tensor.from_numpy(rng.standard_normal(d).astype(np.float16))
    g = S.Graph()
    y = g.add_node("conv", {"x": tensor(3, 3, 38, 42), "w": tensor(16, 3, 7, 7)}, {"size": 7, "activations": 16, "pad": 3, "stride": 2}).y()
    y = g.add_node("batchnorm", {"x": y, **norm_params(rng, 16)}).y()
    y = g.add_node("maxpool", {"x": g.add_node("relu", y).y()}, {"size": 3, "pad": 1, "stride": 2}).y()
    y = g.add_node("concat", {"x0": tensor(3, front, 10, 11), "x1": y, "x2": tensor(3, front, 10, 11)}, {"axis": 1}).y()
    ctx = S.Context()
    p = ctx.create_program(g, 3, training=False)
    ctx.resolve(y)
    p.finalize()
    used = stub_gpu.stub.hipstub_used()
    p.run(2)
    kinds = [op["kind"] for op in stub_gpu.plan(p)]
    assert any(kind.endswith(".pool") for kind in kinds) == (front == 8), kinds
    assert stub_gpu.stub.hipstub_used() == used  # no launch had to ask for any


@pytest.mark.gpu
@pytest.mark.parametrize("look", [["relu"], ["norm"], ["conv"], ["relu", "conv"], ["conv", "relu"]], ids=str)
def test_late_resolved_intermediates(look):
    rng = np.random.default_rng(4)
    x, w = (S.Tensor.from_numpy(rng.standard_normal(d).astype(np.float16)) for d in ((3, 3, 38, 42), (16, 3, 7, 7)))
    norm = norm_params(rng, 16)

    def run(**kwargs):
        g, t = S.Graph(), {}
        t["conv"] = g.add_node("conv", {"x": x, "w": w}, {"size": 7, "activations": 16, "pad": 3, "stride": 2}).y()
        t["norm"] = g.add_node("batchnorm", {"x": t["conv"], **norm}).y()
        t["relu"] = g.add_node("relu", t["norm"]).y()
        t["out"] = g.add_node("maxpool", {"x": t["relu"]}, {"size": 3, "pad": 1, "stride": 2}).y()
        ctx = S.Context()
        p = ctx.create_program(g, 3, training=False, **kwargs)
        return ctx, p, t

    ctx, p, t = run(disable_op_fusing=True)
    want = {k: ctx.resolve(v) for k, v in t.items()}
    p.run(1)
    want = {k: v.read().astype(np.float32) for k, v in want.items()}
    ctx, p, t = run()
    dev = {"out": ctx.resolve(t["out"])}
    for name in [None] + [n for n in look if n in t]:
        if name:
            r = ctx.resolve(t[name])
            if r is None:  # (the norm's own output does not exist: the relu is part of it)
                continue
            dev[name] = r
        p.run(1)
        for k, v in dev.items():
            if k == "norm":
                continue
            np.testing.assert_allclose(v.read().astype(np.float32), want[k], rtol=0, atol=2e-3 * np.abs(want[k]).max())
