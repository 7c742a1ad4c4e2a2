"""The copies of filters that a program keeps between steps (packed fp32, transposed fp16) follow the weights: after host
writes, and after the steps of a training program that shares them."""
import copy

import numpy as np
import pytest

from oracle import ref
from saga_amd import api as S
from saga_amd import networks as N

pytestmark = pytest.mark.gpu


def logits(net, x, weights):
    """A program of its own, built from these weights."""
    net = copy.copy(net)
    net.params = {**net.params, **weights}
    ctx = S.Context()
    g, t = N.build_graph(net, x)
    p = ctx.create_program(g, net.batch, training=False)
    out = ctx.resolve(t[net.output])
    p.run(1)
    return out.read().copy()


@pytest.mark.parametrize("make", [lambda: N.resnet20(4, dtype=S.FLOAT), lambda: N.unet(1, image=32, classes=8, widths=(8, 16, 32, 64),
                                                                                       bottleneck=128)], ids=["fp32", "fp16 transposed"])
def test_host_writes(make):
    net = make()
    rng = np.random.default_rng(1)
    x = rng.standard_normal((net.batch,) + tuple(net.in_shape)).astype(np.float32)
    ctx = S.Context()
    g, t = N.build_graph(net, x)
    p = ctx.create_program(g, net.batch, training=False)
    out = ctx.resolve(t[net.output])
    names = [k for k, v in net.params.items() if v.ndim == 4 and v.shape[2] > 1][-3:]
    dev = {k: ctx.resolve(t[k]) for k in names}
    p.run(1)
    first = out.read().copy()
    p.run(1)
    np.testing.assert_array_equal(out.read(), first)
    for k in names:  # one at a time: each has to be noticed by itself
        new = {k: (net.params[k] * 1.5).astype(np.float32)}
        dev[k].write(new[k])
        p.run(1)
        got = out.read().copy()
        np.testing.assert_array_equal(got, logits(net, x, new))
        assert not np.array_equal(got, first)
        dev[k].write(net.params[k])
        p.run(1)
        np.testing.assert_array_equal(out.read(), first)


def test_training_steps():
    net = N.resnet20(8, dtype=S.FLOAT)
    rng = np.random.default_rng(2)
    x = rng.standard_normal((net.batch,) + tuple(net.in_shape)).astype(np.float32)
    ctx = S.Context()
    g, t = N.build_graph(net, x)
    infer = ctx.create_program(g, net.batch, training=False)
    train = ctx.create_program(g, net.batch, training=True, learning_rate=1e-2)
    ctx.resolve(t["labels"]).write(rng.integers(0, net.classes, (net.batch, 1)).astype(np.int32))
    out = ctx.resolve(t[net.output])
    weights = {k: ctx.resolve(t[k]) for k in net.params}
    for _ in range(3):
        infer.run(1)
        got = out.read().copy()
        np.testing.assert_array_equal(got, logits(net, x, {k: v.read().copy() for k, v in weights.items()}))
        train.run(1)


@pytest.mark.parametrize("transpose", [False, True])
@pytest.mark.parametrize("dtype,other", [(S.FLOAT, S.HALF), (S.HALF, S.FLOAT)], ids=["f32", "f16"])
def test_computed_filter(dtype, other, transpose):
    """A filter that the program itself computes, between two convolutions, is used as this step computed it."""
    rng = np.random.default_rng(3)
    draw = lambda *shape: (rng.standard_normal(shape) / 12).astype(np.float16).astype(N.np_dtype(dtype))
    x, w1 = draw(2, 16, 12, 12), draw(16, 16, 3, 3)
    attrs = {"size": 3, "activations": 16, "pad": 1, "transpose": transpose}

    def conv(g, x, w):
        return g.add_node("conv", {"x": x, "w": w}, attrs).y()

    def program(w2):
        """w2: a front-end tensor's function of the graph."""
        g, ctx = S.Graph(), S.Context()
        y = conv(g, S.Tensor.from_numpy(x), S.Tensor.from_numpy(w1, name="w1"))
        second = w2(g)
        out = conv(g, y, second)
        p = ctx.create_program(g, 2, training=False)
        out = ctx.resolve(out)
        p.finalize()  # places the initial values
        return ctx, p, out

    source = S.Tensor.from_numpy(draw(16, 16, 3, 3).astype(N.np_dtype(other)), name="source")
    ctx, p, out = program(lambda g: g.add_node("convert", {"x": source}, {"datatype": dtype}).y())
    dev = ctx.resolve(source)
    for _ in range(3):
        values = draw(16, 16, 3, 3)
        dev.write(values.astype(N.np_dtype(other)))
        p.run(1)
        _, q, want = program(lambda g: S.Tensor.from_numpy(values, name="w2"))
        q.run(1)
        # the same products, added in another order where the constant filter is packed: fp32 rounding, and in fp16 at most the
        # next value (2^-10 of the largest) where a sum lies between two
        scale = np.abs(want.read()).max()
        assert scale > 0
        np.testing.assert_allclose(out.read() / scale, want.read() / scale, atol=1e-5 if dtype == S.FLOAT else 2e-3)


def test_batched_filter():
    """... and one that the host hands in with every batch."""
    rng = np.random.default_rng(4)
    draw = lambda *shape: rng.standard_normal(shape).astype(np.float32)
    x = draw(2, 16, 12, 12)
    g, ctx = S.Graph(), S.Context()
    w = S.Tensor.from_numpy(draw(16, 16, 3, 3), name="w")
    out = g.add_node("conv", {"x": S.Tensor.from_numpy(x), "w": w}, {"size": 3, "activations": 16, "pad": 1}).y()
    p = ctx.create_program(g, 2, training=False, batched={w: S.PRE})
    out, dev = ctx.resolve(out), ctx.resolve(w)
    p.finalize()
    for _ in range(3):
        values = draw(16, 16, 3, 3)
        dev.write(values)
        p.run(1)
        want = ref.conv2d_fwd(x, values, 1, 1)
        np.testing.assert_allclose(out.read() / np.abs(want).max(), want / np.abs(want).max(), atol=1e-5)
