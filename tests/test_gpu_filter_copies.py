"""The copies of filters that a program keeps between steps (packed fp32, transposed fp16) follow the weights: after host
writes, and after the steps of a training program that shares them."""
import copy

import numpy as np
import pytest

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
