"""Inference programs fold norms and relus into the operations in front of them.  Whoever looks at a tensor that went that way
- the host before or after the program is finalized, another view, another program - still finds its values."""
import numpy as np
import pytest

from saga_amd import api as S
from saga_amd import networks as N
from tests.test_engine_plan import FOLDED, chain, norm_params

pytestmark = pytest.mark.gpu

# of the largest value: fp32 sums in another order; up to four roundings to fp16 (2^-11 each) on the way to an output
TOL = {S.FLOAT: 1e-5, S.HALF: 2e-3}


def close(got, want, dtype):
    assert np.abs(want).max() > 0
    np.testing.assert_allclose(got.astype(np.float32) / np.abs(want).max(), want.astype(np.float32) / np.abs(want).max(), rtol=0, atol=TOL[dtype])


def unfused(dtype):
    """Every tensor of the chain by its own operation."""
    g, t = chain(dtype)
    ctx = S.Context()
    p = ctx.create_program(g, 2, training=False, disable_op_fusing=True)
    dev = {k: ctx.resolve(v) for k, v in t.items()}
    p.run(1)
    return {k: v.read().copy() for k, v in dev.items()}


@pytest.mark.parametrize("when", ["before finalize", "between steps"])
@pytest.mark.parametrize("dtype", [S.FLOAT, S.HALF], ids=["f32", "f16"])
def test_late_resolved_intermediates(dtype, when):
    want = unfused(dtype)
    g, t = chain(dtype)
    ctx = S.Context()
    p = ctx.create_program(g, 2, training=False)
    dev = {"out": ctx.resolve(t["out"])}
    for name in FOLDED[dtype] + ["relu", "norm"]:
        if when == "between steps":
            p.run(1)
        dev[name] = ctx.resolve(t[name])
        if when == "between steps":
            p.run(1)
            for k, v in dev.items():
                close(v.read(), want[k], dtype)
    p.run(1)
    for k, v in dev.items():
        close(v.read(), want[k], dtype)


@pytest.mark.parametrize("fused", [True, False])
def test_late_resolve_under_graphs(fused, monkeypatch):
    """Recorded launches are recorded again for the longer list."""
    monkeypatch.setenv("SAGA_HIP_GRAPH", "1")
    net = N.resnet20(4, dtype=S.FLOAT)
    x = np.random.default_rng(3).standard_normal((4,) + tuple(net.in_shape)).astype(np.float32)
    g, t = N.build_graph(net, x, with_classifier=False)
    ctx = S.Context()
    p = ctx.create_program(g, 4, training=False, disable_op_fusing=not fused)
    out = ctx.resolve(t[net.output])
    p.run(4)
    first = out.read().copy()
    conv = ctx.resolve(t[net.nodes[0]["out"]])
    for _ in range(3):
        p.run(2)
        np.testing.assert_allclose(out.read(), first, rtol=0, atol=1e-5 * np.abs(first).max())
        assert np.abs(conv.read()).max() > 0


def test_late_resolve_of_several_folds_under_graphs(monkeypatch):
    """The stem's convolution has its norm and its pooling: both come back, and what is between them has memory before it is recorded."""
    net = N.resnet50(2, dtype=S.HALF, image=64)
    x = np.random.default_rng(3).standard_normal((2,) + tuple(net.in_shape)).astype(np.float16)
    seen = []
    for graphs in ("0", "1"):
        monkeypatch.setenv("SAGA_HIP_GRAPH", graphs)
        g, t = N.build_graph(net, x, with_classifier=False)
        ctx = S.Context()
        p = ctx.create_program(g, 2, training=False)
        out = ctx.resolve(t[net.output])
        p.run(4)
        seen.append([out.read().copy()])
        conv = ctx.resolve(t[net.nodes[0]["out"]])
        for _ in range(3):
            p.run(2)
            seen[-1] += [out.read().copy(), conv.read().copy()]
    for a, b in zip(*seen):
        assert np.abs(a).max() > 0 and np.array_equal(a, b)


def test_residual_behind_the_convolution_and_a_window():
    rng = np.random.default_rng(2)
    draw = lambda *shape: S.Tensor.from_numpy(rng.standard_normal(shape).astype(np.float32))
    x, w, w1, norm = draw(2, 16, 6, 6), draw(16, 16, 3, 3), draw(16, 16, 1, 1), norm_params(rng, 16)

    def run(**kwargs):
        g = S.Graph()
        main = g.add_node("conv", {"x": x, "w": w}, {"size": 3, "activations": 16, "pad": 1}).y()
        side = g.add_node("sigmoid", g.add_node("conv", {"x": x, "w": w1}, {"size": 1, "activations": 16})).y()
        n = g.add_node("batchnorm", {"x": main, **norm}).y()
        a = g.add_node("relu", g.add_node("sum", {"x0": n, "x1": side})).y()
        other = g.add_node("conv", {"x": x, "w": w1}, {"size": 1, "activations": 16}).y()
        b = g.add_node("batchnorm", {"x": other, **norm}).y()
        c = g.add_node("sigmoid", g.add_node("window", {"x": other}, {"offset": [0, 4, 0, 0], "shape": [2, 8, 6, 6]})).y()
        ctx = S.Context()
        p = ctx.create_program(g, 2, training=False, **kwargs)
        out = [ctx.resolve(v) for v in (a, b, c)]
        p.run(1)
        return [v.read().copy() for v in out]

    for got, want in zip(run(), run(disable_op_fusing=True)):
        close(got, want, S.FLOAT)


def test_late_resolve_inside_a_recorded_run(monkeypatch):
    """What a folded operation wrote gets its memory when somebody asks for it, not between the launches that are recorded."""
    monkeypatch.setenv("SAGA_HIP_GRAPH", "1")
    net = N.resnet20(4, dtype=S.FLOAT)
    x = np.random.default_rng(3).standard_normal((4,) + tuple(net.in_shape)).astype(np.float32)
    g, t = N.build_graph(net, x, with_classifier=False)
    ctx = S.Context()
    p = ctx.create_program(g, 4, training=False)
    out = ctx.resolve(t[net.output])
    p.run(4)
    first = out.read().copy()
    conv = ctx.resolve(t[[n for n in net.nodes if n["type"] == "conv"][9]["out"]])
    for _ in range(3):
        p.run(2)
        np.testing.assert_allclose(out.read(), first, rtol=0, atol=1e-5 * np.abs(first).max())
        assert np.abs(conv.read()).max() > 0
