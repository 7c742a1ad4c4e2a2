"""fp32 convolutions with a max pooling of 2x2 windows in their epilogue: which calls have one, held on the stub runtime; on the GPU
against the convolution and the pooling by themselves."""
import ctypes as C

import numpy as np
import pytest
import torch

from saga_amd import api as S
from saga_amd import kernels as K
from saga_amd import networks as N
from tests import stub_gpu
from tests.stub_gpu import on_stub

# N, C, H, W, K, filter, pad, stride: kernel
SHAPES = {
    (64, 1, 28, 28, 32, 5, 2, 1): "stream_f32_k_thin",
    (3, 1, 28, 28, 20, 5, 0, 1): "stream_f32_k_thin",       # channels in part of a block, the last tile in part
    (2, 3, 31, 45, 70, 3, 1, 1): "stream_f32_k_thin",       # odd sizes: a row and a column without a window
    (160, 3, 33, 29, 64, 7, 3, 2): "stream_f32_k_thin",
    (1, 4, 2, 3, 8, 3, 1, 1): "stream_f32_k_thin",          # one window
    (64, 32, 14, 14, 64, 5, 2, 1): "stream_f32_k_window",
    (61, 32, 15, 17, 40, 5, 2, 1): "stream_f32_k_window",
    (90, 64, 28, 28, 72, 3, 1, 1): "stream_f32_k_window",
    (37, 24, 29, 31, 130, 3, 1, 1): "stream_f32_k_window",
    (50, 16, 20, 23, 32, 3, 2, 1): "stream_f32_k_window",   # more pixels than positions
    (4, 64, 14, 14, 64, 5, 2, 1): None,                     # a grid that needs its reduction split
    (64, 64, 28, 28, 64, 1, 0, 1): None,
    (16, 64, 70, 70, 64, 3, 1, 1): None,                    # long rows
    (64, 64, 28, 28, 64, 3, 1, 2): None,
}


def dims(shape):
    n, c, h, w, k, r, pad, stride = shape
    p, q = ((e + 2 * pad - r) // stride + 1 for e in (h, w))
    return (n, c, h, w), (k, c, r, r), (n, k, p, q), (n, k, p // 2, q // 2), K.ConvParams(pad, stride, 1, 1)


def extras(bias=None, norm=None, relu=1, packed=None):
    e = K.ConvExtras(relu=relu)
    if bias is not None:
        e.bias = C.pointer(bias)
    if norm is not None:
        e.s, e.b, e.m, e.v = norm
        e.eps = 1e-3
    if packed is not None:
        e.packed = packed
    return e


@on_stub
def test_routes():
    L = K.lib()
    for shape, kernel in SHAPES.items():
        xs, ws, _, ys, p = dims(shape)
        x, w, y = (K.TensorView() for _ in range(3))
        for v, d, at in ((x, xs, 20), (w, ws, 30), (y, ys, 31)):
            v.ptr, v.dtype, v.dims[:] = 1 << at, K.FLOAT, d
            v.strides[:] = torch.empty(d, device="meta").stride()
        X, W, Y, P, e = (C.byref(a) for a in (x, w, y, p, extras(relu=1)))
        ok = L.saga_hip_conv2d_fwd_maxpool_ok(X, W, Y, P, e, 2, 0, 2)
        assert bool(ok) == (kernel is not None), shape
        for pool in ((3, 0, 2), (2, 0, 1), (2, 1, 2)):
            assert not L.saga_hip_conv2d_fwd_maxpool_ok(X, W, Y, P, e, *pool)
        stub_gpu.launched()
        rc = L.saga_hip_conv2d_fwd_maxpool(X, W, Y, P, e, 2, 0, 2, 1 << 32, 1 << 28, None)
        ran = [name for name, *_ in stub_gpu.launched()]
        assert (rc == 0) == (kernel is not None) and (ran[-1:] == [kernel] if kernel else ran == []), (shape, ran)
        if kernel == "stream_f32_k_window":  # without room to pack the filter there is none
            assert L.saga_hip_conv2d_fwd_maxpool(X, W, Y, P, e, 2, 0, 2, 1 << 32, 1024, None) != 0 and stub_gpu.launched() == []


@on_stub
def test_the_digits_classifier():
    net = N.lenet(64)
    g, t = N.build_graph(net, np.zeros((64, 1, 28, 28), np.float32), with_classifier=False)
    ctx = S.Context()
    p = ctx.create_program(g, 64, training=False)
    ctx.resolve(t[net.output])
    p.finalize()
    kinds = [op["kind"] for op in stub_gpu.plan(p) if op["kind"] != "filterpack"]
    assert kinds == ["convfwd.pool", "convfwd.pool", "fc.fwd.n", "fc.fwd.n"]
    for n in net.nodes:  # and back again, the pooling first
        ctx.resolve(t[n["out"]])
    kinds = [op["kind"] for op in stub_gpu.plan(p) if op["kind"] != "filterpack"]
    assert kinds == ["convfwd", "actfwd", "poolfwd"] * 2 + ["fc.fwd.n", "actfwd", "fc.fwd.n"]


def pooled_then_normalised(behind, **config):
    """conv -> max pooling -> batch norm or relu, and the result."""
    rng = np.random.default_rng(5)
    tensor = lambda a: S.Tensor.from_numpy(a.astype(np.float32))
    g = S.Graph()
    x, w = tensor(rng.standard_normal((64, 1, 28, 28))), tensor(rng.standard_normal((32, 1, 5, 5)) / 5)
    y = g.add_node("conv", {"x": x, "w": w}, {"size": 5, "activations": 32, "pad": 2}).y()
    y = g.add_node("maxpool", {"x": y}, {"size": 2, "stride": 2}).y()
    if behind == "norm":  # (scales of either sign: a norm and a pooling do not change places)
        params = {k: tensor(rng.standard_normal((1, 32)) if k != "v" else rng.uniform(0.5, 1.5, (1, 32))) for k in "sbmv"}
        y = g.add_node("batchnorm", {"x": y, **params}).y()
    else:
        y = g.add_node(behind, {"x": y}).y()
    ctx = S.Context()
    p = ctx.create_program(g, 64, training=False, **config)
    return p, ctx.resolve(y)


@on_stub
def test_a_norm_behind_the_pooling_stays_there():
    for behind, want in (("norm", ["convfwd.pool", "bninf"]), ("relu", ["convfwd", "poolfwd"])):
        p, _ = pooled_then_normalised(behind)
        p.finalize()
        ops = [op for op in stub_gpu.plan(p) if op["kind"] != "filterpack"]
        assert [op["kind"] for op in ops] == want


@pytest.mark.gpu
@pytest.mark.parametrize("behind", ["norm", "relu"])
def test_what_is_behind_the_pooling(behind):
    got = []
    for fused in (True, False):
        p, out = pooled_then_normalised(behind, disable_op_fusing=not fused)
        p.run(1)
        got.append(out.read().copy())
    assert np.abs(got[1]).max() > 0
    np.testing.assert_allclose(*got, rtol=0, atol=1e-5 * np.abs(got[1]).max())


@pytest.mark.parametrize("shape", [s for s, k in SHAPES.items() if k and s[0] > 1], ids=str)
@on_stub
def test_an_output_out_of_reach(shape):
    """Pooled results that are part of a tensor of more than 2 GiB: no such launch, and asked beforehand there is none either."""
    L = K.lib()
    xs, ws, _, ys, p = dims(shape)
    x, w, y = (K.TensorView() for _ in range(3))
    for v, d, at in ((x, xs, 20), (w, ws, 30), (y, ys, 31)):
        v.ptr, v.dtype, v.dims[:] = 1 << at, K.FLOAT, d
        v.strides[:] = torch.empty(d, device="meta").stride()
    y.strides[0] = (1 << 29) // (ys[0] - 1)
    X, W, Y, P, e = (C.byref(a) for a in (x, w, y, p, extras(relu=1)))
    assert L.saga_hip_conv2d_fwd_maxpool(X, W, Y, P, e, 2, 0, 2, 1 << 33, 1 << 30, None) == -3
    assert not L.saga_hip_conv2d_fwd_maxpool_ok(X, W, Y, P, e, 2, 0, 2)


@pytest.mark.gpu
@pytest.mark.parametrize("what", ["bias", "norm", "nothing", "not finite"])
@pytest.mark.parametrize("shape", [s for s, k in SHAPES.items() if k], ids=str)
def test_against_both(shape, what):
    xs, ws, us, ys, p = dims(shape)
    g = torch.Generator("cuda").manual_seed(sum(xs))
    draw = lambda d, by=1.0: torch.randn(d, device="cuda", generator=g) / by
    x, w = draw(xs), draw(ws, (ws[1] * ws[2] * ws[3]) ** 0.5)
    if what == "not finite":
        x[0, 0, 0, 0], x[-1, -1, -1, -1] = float("nan"), float("-inf")
    bias = draw((1, ws[0], 1, 1))
    norm = [draw((ws[0],)) for _ in range(3)] + [torch.rand(ws[0], device="cuda", generator=g) + 0.5]  # (scales of either sign)
    L, V = K.lib(), lambda t: K.view(t)
    vx, vw, vb = V(x), V(w), V(bias)
    between = torch.empty(us, device="cuda")
    want = torch.empty(ys, device="cuda")
    room = torch.full((ys[0], ys[1] + 2, ys[2] + 3, ys[3] + 1), 7.0, device="cuda")
    got = room[:, 1:1 + ys[1], 2:2 + ys[2], :ys[3]]
    vu, vo, vg = V(between), V(want), V(got)
    P = C.byref(p)
    n = L.saga_hip_conv2d_workspace_size(K.CONV_FWD, C.byref(vx), C.byref(vw), C.byref(vu), P)
    space = torch.empty(max(n, 16), dtype=torch.uint8, device="cuda")
    e = extras(vb) if what in ("bias", "not finite") else extras(norm=[t.data_ptr() for t in norm]) if what == "norm" else extras(relu=0)
    st = K.stream_ptr()
    K.check(L.saga_hip_conv2d_fwd_ex(C.byref(vx), C.byref(vw), C.byref(vu), P, 0.0, C.byref(e), K.ptr(space), space.numel(), st))
    K.check(L.saga_hip_pool_fwd(K.POOL_MAX, C.byref(vu), C.byref(vo), None, 2, 0, 2, st))
    assert L.saga_hip_conv2d_fwd_maxpool_ok(C.byref(vx), C.byref(vw), C.byref(vg), P, C.byref(e), 2, 0, 2)
    K.check(L.saga_hip_conv2d_fwd_maxpool(C.byref(vx), C.byref(vw), C.byref(vg), P, C.byref(e), 2, 0, 2, K.ptr(space), space.numel(), st))
    ok = torch.isfinite(want)
    assert torch.equal(torch.isfinite(got), ok) and torch.equal(torch.isnan(got), torch.isnan(want))
    # the same products in the same order, unless the convolution alone splits its reduction: then sums in another order
    scale = torch.where(ok, want, 0.0).abs().max()
    assert torch.where(ok, got - want, 0.0).abs().max() <= 1e-5 * scale and (scale > 0 or what == "not finite")
    got.fill_(7.0)
    assert (room == 7.0).all()  # nothing beside the result


@pytest.mark.gpu
def test_a_late_look_at_what_is_between():
    net = N.lenet(50)
    x = np.random.default_rng(3).random((50, 1, 28, 28)).astype(np.float32)
    runs = []
    for fused in (False, True):
        g, t = N.build_graph(net, x, with_classifier=False)
        ctx = S.Context()
        p = ctx.create_program(g, 50, training=False, disable_op_fusing=not fused)
        out = ctx.resolve(t[net.output])
        seen = []
        for n in net.nodes[:-1]:
            p.run(1)
            seen.append(out.read().copy())
            d = ctx.resolve(t[n["out"]])
            p.run(1)
            seen.append(d.read().copy())
        runs.append(seen)
    for a, b in zip(*runs):
        assert np.abs(a).max() > 0
        np.testing.assert_allclose(a, b, rtol=0, atol=1e-5 * np.abs(a).max())
