"""What the engine plans for a program, looked at without a GPU: which memory the operations share, and in which order the two
streams run those that do."""
import numpy as np
import pytest

from saga_amd import api as S
from saga_amd import networks as N
from tests import stub_gpu
from tests.stub_gpu import on_stub


def behind_resize(net, image, pixels=None):
    """The training graph of `net` behind byte images that are converted and resized to the network's input, and its tensors."""
    g = S.Graph()
    if pixels is None:
        pixels = S.Tensor.placeholder(S.U8, [net.batch, 3, image, image], "pixels")
    c = g.add_node("convert", {"x": pixels}, {"scale": 1 / 255.0, "datatype": net.dtype})
    c = g.add_node("spatialtransform", {"x": c.y()}, {"height": net.in_shape[1], "width": net.in_shape[2]})
    t = {net.input: c.y()}
    for name, a in net.params.items():
        norm = name.endswith(("-s", "-m", "-v")) or name[:-2] + "-s" in net.params
        t[name] = S.Tensor.from_numpy(a.astype(N.np_dtype(S.FLOAT if norm else net.dtype)), name=name)
    for n in net.nodes:
        t[n["out"]] = g.add_node(n["type"], {k: t[v] for k, v in n["in"].items()}, n["attrs"], n["name"]).y()
    head = g.add_node("catclassifier", {"x": t[net.output]})
    t["loss"], t["labels"] = head.output("loss"), head.y().grad()
    return g, t


TRAINED = {
    "resnet20": lambda: N.resnet20(64),
    "resnet20 f32": lambda: N.resnet20(64, dtype=S.FLOAT),
    "resnet50": lambda: N.resnet50(16, image=128),
    "lenet": lambda: N.lenet(64),
    "unet": lambda: N.unet(2, image=64),
}


@pytest.mark.parametrize("name", TRAINED)
@on_stub
def test_operations_that_share_memory_are_ordered(name):
    net = TRAINED[name]()
    if name == "unet":  # a scalar loss
        b = N.Builder(net, 99)
        b.shape[net.output] = (net.classes, 64, 64)
        net.output = b.fc(b.pool("avgpool", net.output, global_=True), "cls", net.classes)
    ctx = S.Context()
    g, _ = N.build_graph(net, np.zeros((net.batch,) + tuple(net.in_shape), np.float32))
    p = ctx.create_program(g, net.batch, training=True)
    p.finalize()
    ops = stub_gpu.plan(p)
    assert any(op["side"] for op in ops)
    bad = stub_gpu.unordered(ops)
    assert not bad, bad[:8]


@pytest.mark.parametrize("name,image", [("resnet20", 512), ("resnet50", 1024)])
@on_stub
def test_operations_in_front_of_the_first_convolution_are_ordered(name, image):
    """Their tensors are large and done with early: what the side stream writes from the start of the step must stay out of
    that memory."""
    net = TRAINED[name]()
    ctx = S.Context()
    p = ctx.create_program(behind_resize(net, image)[0], net.batch, training=True)
    p.finalize()
    ops = stub_gpu.plan(p)
    kinds = [op["kind"] for op in ops]
    assert kinds[:2] == ["convert", "spatialtransform"] and "filtertranspose" in [op["kind"] for op in ops if op["side"]]
    bad = stub_gpu.unordered(ops)
    assert not bad, bad[:8]


def computed_filters(dtype, other, transpose):
    """conv(x, w1), w2 = convert(w2h), conv(y, w2): a filter that the program computes between two convolutions."""
    rng = np.random.default_rng(1)
    g = S.Graph()
    half = lambda shape: rng.standard_normal(shape).astype(np.float16)
    x = S.Tensor.from_numpy(half((2, 16, 12, 12)).astype(N.np_dtype(dtype)))
    w1 = S.Tensor.from_numpy(half((16, 16, 3, 3)).astype(N.np_dtype(dtype)), name="w1")
    w2h = S.Tensor.from_numpy(half((16, 16, 3, 3)).astype(N.np_dtype(other)), name="w2h")
    attrs = {"size": 3, "activations": 16, "pad": 1, "transpose": transpose}
    y = g.add_node("conv", {"x": x, "w": w1}, attrs).y()
    w2 = g.add_node("convert", {"x": w2h}, {"datatype": dtype}).y()
    return g, w2h, g.add_node("conv", {"x": y, "w": w2}, attrs).y()


@pytest.mark.parametrize("transpose", [False, True])
@pytest.mark.parametrize("dtype,other", [(S.FLOAT, S.HALF), (S.HALF, S.FLOAT)], ids=["f32", "f16"])
@on_stub
def test_computed_filters_are_not_copied_beforehand(dtype, other, transpose):
    g, _, out = computed_filters(dtype, other, transpose)
    ctx = S.Context()
    p = ctx.create_program(g, 2, training=False)
    ctx.resolve(out)
    p.finalize()
    ops = stub_gpu.plan(p)
    convert, = [i for i, op in enumerate(ops) if op["kind"] == "convert"]
    (filter2, *_), = ops[convert]["writes"]
    early = [op["kind"] for op in ops[:convert] for s, *_ in op["reads"] if s == filter2]
    assert not early, early
    # the filter that nothing computes still has its copy, where its kernel reads one
    copies = [op for op in ops if op["kind"] in ("filterpack", "filtertranspose")]
    assert len(copies) == (0 if dtype == S.HALF and not transpose else 1)
    assert all(len(op["reads"]) == 1 for op in copies)


@on_stub
def test_batched_filters_are_not_copied():
    """A batched tensor's contents and address change under the operations."""
    g = S.Graph()
    x = S.Tensor.from_numpy(np.zeros((2, 16, 12, 12), np.float32))
    w = S.Tensor.from_numpy(np.zeros((16, 16, 3, 3), np.float32), name="w")
    out = g.add_node("conv", {"x": x, "w": w}, {"size": 3, "activations": 16, "pad": 1}).y()
    ctx = S.Context()
    p = ctx.create_program(g, 2, training=False, batched={w: S.PRE})
    ctx.resolve(out)
    p.finalize()
    assert [op["kind"] for op in stub_gpu.plan(p)] == ["convfwd"]


def batched_relu():
    g = S.Graph()
    x = S.Tensor.from_numpy(np.zeros((2, 8), np.float32), name="x")
    y = g.add_node("relu", {"x": x}).y()
    ctx = S.Context()
    p = ctx.create_program(g, 2, training=False, batched={x: S.PRE})
    return p, ctx.resolve(x), ctx.resolve(y)


@pytest.mark.parametrize("steps", [1, 2])
@on_stub
def test_a_pointer_kept_over_steps_is_uploaded(steps):
    """The access object and the pointer are asked for once, the values are written before every run."""
    p, x, _ = batched_relu()
    p.finalize()
    window = stub_gpu.Window(x)
    data = window.floats(16)
    for value in (1, 2, 3, 4):
        data[:] = value
        p.run(steps)
        if steps == 1:  # (an even number of steps leaves the other buffer behind)
            np.testing.assert_array_equal(stub_gpu.last_batch(x, 16), value)
    data[:] = 5
    window.close()  # what was written before the window was closed counts
    p.run(1)
    seen = [stub_gpu.last_batch(x, 16)[0]]
    p.run(2)
    seen.append(stub_gpu.last_batch(x, 16)[0])
    assert 5 in seen, seen


@on_stub
def test_untouched_batches_are_uploaded_once():
    p, x, _ = batched_relu()
    p.finalize()
    before = stub_gpu.uploads()
    x.write(np.ones((2, 8), np.float32))
    p.run(1)
    assert stub_gpu.uploads() - before == 1
    np.testing.assert_array_equal(stub_gpu.last_batch(x, 16), 1)
    p.run(1)
    assert stub_gpu.uploads() - before == 1


def norm_params(rng, c):
    return {k: S.Tensor.from_numpy(rng.uniform(0.5, 1.5, (1, c)).astype(np.float32), name="bn-" + k) for k in "sbmv"}


def chain(dtype):
    """conv + bias -> relu -> maxpool -> relu -> conv -> batch norm -> sigmoid, and its intermediate tensors by name."""
    rng = np.random.default_rng(2)
    draw = lambda *shape, by=1: S.Tensor.from_numpy((rng.standard_normal(shape) / by).astype(N.np_dtype(dtype)))
    g, t = S.Graph(), {}
    attrs = {"size": 3, "activations": 16, "pad": 1}
    t["conv"] = g.add_node("conv", {"x": draw(2, 16, 12, 12), "w": draw(16, 16, 3, 3, by=12), "b": draw(1, 16)}, {**attrs, "bias": True}).y()
    t["relu"] = g.add_node("relu", {"x": t["conv"]}).y()
    t["pool"] = g.add_node("maxpool", {"x": t["relu"]}, {"size": 2, "stride": 2}).y()
    t["relu2"] = g.add_node("relu", {"x": t["pool"]}).y()
    t["conv2"] = g.add_node("conv", {"x": t["relu2"], "w": draw(16, 16, 3, 3, by=12)}, attrs).y()
    t["norm"] = g.add_node("batchnorm", {"x": t["conv2"], **norm_params(rng, 16)}).y()
    t["out"] = g.add_node("sigmoid", {"x": t["norm"]}).y()
    return g, t


FOLDED = {S.FLOAT: ["conv", "pool", "conv2"], S.HALF: ["pool", "conv2"]}


def written(ops):
    return [s for op in ops for s, *_ in op["writes"]]


@pytest.mark.parametrize("dtype", [S.FLOAT, S.HALF], ids=["f32", "f16"])
@on_stub
def test_what_nobody_looks_at_is_folded_away(dtype):
    g, t = chain(dtype)
    ctx = S.Context()
    p = ctx.create_program(g, 2, training=False)
    ctx.resolve(t["out"])
    p.finalize()
    kinds = [op["kind"] for op in stub_gpu.plan(p) if op["kind"] != "filterpack"]
    assert kinds == {S.FLOAT: ["convfwd", "poolfwd", "convfwd.bn", "actfwd"],
                     S.HALF: ["convfwd", "actfwd", "poolfwd", "convfwd.bn", "actfwd"]}[dtype]


@pytest.mark.parametrize("finalized", [False, True], ids=["behind create_program", "behind finalize"])
@pytest.mark.parametrize("dtype", [S.FLOAT, S.HALF], ids=["f32", "f16"])
@on_stub
def test_resolved_intermediates_are_written(dtype, finalized):
    """Also when they are resolved late, one after the other: each is an operation's output then, and all that was written before
    still is, in an order that suits the readers."""
    g, t = chain(dtype)
    ctx = S.Context()
    p = ctx.create_program(g, 2, training=False, anomaly_detect=True)
    ctx.resolve(t["out"])
    if finalized:
        p.finalize()
        before = stub_gpu.plan(p)
        outputs = {s for op in before for s, *_ in op["writes"]}
    for n, name in enumerate(FOLDED[dtype]):
        assert ctx.resolve(t[name]) is not None
        if finalized:
            ops = stub_gpu.plan(p)
            assert len(ops) == len(before) + n + 1
            assert outputs < set(written(ops))
    p.run(1)
    ops = stub_gpu.plan(p)
    assert [op["kind"] for op in ops if op["kind"] != "filterpack"] == ["convfwd", "actfwd", "poolfwd", "actfwd", "convfwd", "bninf", "actfwd"]
    seen = written(ops)
    assert len(seen) == len(set(seen))
    for i, op in enumerate(ops):  # no operation reads what a later one writes
        later = set(written(ops[i:]))
        assert not [s for s, *_ in op["reads"] if s in later]
    assert stub_gpu.unordered(ops) == [] and stub_gpu.overlapping(ops) == []


def nothing_without_memory(p):
    """(memory that nobody has asked for yet would be allocated by a launch, which may be one that is recorded)"""
    return all(address for op in stub_gpu.plan(p) for _, address, *_ in op["reads"] + op["writes"])


@pytest.mark.parametrize("name", ["lenet", "resnet50"])
@on_stub
def test_what_is_written_again_has_memory(name):
    """Of several operations that are folded into one, all come back with the first: also the tensors between the others."""
    net = N.lenet(64) if name == "lenet" else N.resnet50(1, dtype=S.HALF)
    g, t = N.build_graph(net, np.zeros((net.batch,) + tuple(net.in_shape), np.float32), with_classifier=False)
    ctx = S.Context()
    p = ctx.create_program(g, net.batch, training=False)
    ctx.resolve(t[net.output])
    p.run(3)
    assert nothing_without_memory(p)
    count = len(stub_gpu.plan(p))
    ctx.resolve(t[net.nodes[0]["out"]])
    assert len(stub_gpu.plan(p)) == count + 2 and nothing_without_memory(p)


@pytest.mark.parametrize("arena", [True, False])
@on_stub
def test_what_another_program_brings_back_has_memory(arena):
    import os

    if not arena:
        os.environ["SAGA_HIP_NO_ARENA"] = "1"
    net = N.lenet(64)
    g, t = N.build_graph(net, np.zeros((64,) + tuple(net.in_shape), np.float32), with_classifier=False)
    ctx = S.Context()
    p = ctx.create_program(g, 64, training=False)
    ctx.resolve(t[net.output])
    p.run(3)
    count = len(stub_gpu.plan(p))
    h = S.Graph()
    ctx_out = h.add_node("tanh", {"x": t[net.nodes[0]["out"]]}).y()
    q = ctx.create_program(h, 64, training=False)
    ctx.resolve(ctx_out)
    q.finalize()
    assert len(stub_gpu.plan(p)) == count + 2 and nothing_without_memory(p)


@on_stub
def test_a_window_onto_an_intermediate_keeps_it():
    """Other views of the same storage read it too."""
    rng = np.random.default_rng(2)
    draw = lambda *shape: S.Tensor.from_numpy(rng.standard_normal(shape).astype(np.float32))
    g = S.Graph()
    y = g.add_node("conv", {"x": draw(2, 8, 6, 6), "w": draw(16, 8, 3, 3)}, {"size": 3, "activations": 16, "pad": 1}).y()
    a = g.add_node("batchnorm", {"x": y, **norm_params(rng, 16)}).y()
    b = g.add_node("sigmoid", g.add_node("window", {"x": y}, {"offset": [0, 4, 0, 0], "shape": [2, 8, 6, 6]})).y()
    ctx = S.Context()
    p = ctx.create_program(g, 2, training=False)
    ctx.resolve(a), ctx.resolve(b)
    p.finalize()
    ops = [op for op in stub_gpu.plan(p) if op["kind"] != "filterpack"]
    assert sorted(op["kind"] for op in ops) == ["actfwd", "bninf", "convfwd"]


@pytest.mark.parametrize("training", [False, True])
@pytest.mark.parametrize("view", ["window", "concat"])
@on_stub
def test_views_of_a_norms_output_keep_it(view, training):
    """A norm and the relu behind it are one operation, unless a view looks at what is between them."""
    rng = np.random.default_rng(2)
    draw = lambda *shape: S.Tensor.from_numpy(rng.standard_normal(shape).astype(np.float32), name=f"p{rng.integers(1 << 40)}")
    g = S.Graph()
    x = draw(2, 16, 6, 6)
    y = g.add_node("conv", {"x": x, "w": draw(16, 16, 3, 3)}, {"size": 3, "activations": 16, "pad": 1}).y()
    n = g.add_node("batchnorm", {"x": y, **norm_params(rng, 16)}).y()
    a = g.add_node("relu", {"x": n}).y()
    if view == "window":
        b = g.add_node("window", {"x": n}, {"offset": [0, 0, 0, 0], "shape": [2, 16, 6, 6]}).y()
    else:
        other = g.add_node("conv", {"x": x, "w": draw(8, 16, 1, 1)}, {"size": 1, "activations": 8}).y()
        b = g.add_node("concat", {"x0": n, "x1": other}, {"axis": 1}).y()
    b = g.add_node("conv", {"x": b, "w": draw(16, 16 if view == "window" else 24, 1, 1)}, {"size": 1, "activations": 16}).y()
    s = g.add_node("sum", {"x0": a, "x1": b}).y()
    out = g.add_node("fc", {"x": g.add_node("avgpool", {"x": s}, {"global": True}).y(), "w": draw(16, 10)}, {"outputs": 10}).y()
    if training:
        g.add_node("catclassifier", {"x": out})
    ctx = S.Context()
    p = ctx.create_program(g, 2, training=training)
    ctx.resolve(out)
    p.finalize()
    ops = [op for op in stub_gpu.plan(p) if op["kind"] != "filterpack"]
    kinds = [op["kind"] for op in ops]
    norm = kinds.index("bntrain" if training else "convfwd.bn")
    assert "actfwd" in kinds[norm:]
    (between, *_), = [w for w in ops[norm]["writes"] if w[3] == "y"]
    readers = [op["kind"] for op in ops[norm + 1:] for s, *_ in op["reads"] if s == between]
    assert "actfwd" in readers and "convfwd" in readers


@on_stub
def test_a_residual_that_is_computed_behind_the_convolution():
    """The addition cannot move in front of what it adds."""
    rng = np.random.default_rng(2)
    draw = lambda *shape: S.Tensor.from_numpy(rng.standard_normal(shape).astype(np.float32))
    g = S.Graph()
    x = draw(2, 16, 6, 6)
    main = g.add_node("conv", {"x": x, "w": draw(16, 16, 3, 3)}, {"size": 3, "activations": 16, "pad": 1}).y()
    side = g.add_node("conv", {"x": x, "w": draw(16, 16, 1, 1)}, {"size": 1, "activations": 16}).y()
    side = g.add_node("sigmoid", {"x": side}).y()
    norm = g.add_node("batchnorm", {"x": main, **norm_params(rng, 16)}).y()
    out = g.add_node("relu", g.add_node("sum", {"x0": norm, "x1": side})).y()
    ctx = S.Context()
    p = ctx.create_program(g, 2, training=False)
    ctx.resolve(out)
    p.finalize()
    ops = stub_gpu.plan(p)
    (sigmoid, *_), = [op["writes"][0] for op in ops if op["kind"] == "actfwd"]
    place = [op["kind"] for op in ops].index("actfwd")
    assert all(sigmoid not in [s for s, *_ in op["reads"]] for op in ops[:place])


@on_stub
def test_another_program_reads_an_intermediate():
    """A program that starts from what another one computes on the way."""
    g, t = chain(S.FLOAT)
    ctx = S.Context()
    p = ctx.create_program(g, 2, training=False)
    ctx.resolve(t["out"])
    p.finalize()
    h = S.Graph()
    outs = [h.add_node("tanh", {"x": t[k]}).y() for k in ("conv2", "relu", "norm")]
    q = ctx.create_program(h, 2, training=False)
    for v in outs:
        ctx.resolve(v)
    q.finalize()
    ops = stub_gpu.plan(p)
    sources = [op["reads"][0] for op in stub_gpu.plan(q)]
    assert {s for s, *_ in sources} <= set(written(ops))
    # what it starts from shares memory with nothing: p runs to its end in between
    for s, a, size, _ in sources:
        for other, b, n, _ in [x for op in ops + stub_gpu.plan(q) for x in op["reads"] + op["writes"]]:
            assert other == s or not a or not b or a + size <= b or b + n <= a


@pytest.mark.parametrize("with_inference", [False, True], ids=["training alone", "training and inference"])
@pytest.mark.parametrize("name", ["lenet", "resnet20", "resnet20 behind large images"])
@on_stub
def test_what_fits_on_one_stream_fits(name, with_inference):
    """The second stream is given up where memory is short, and only there."""
    import gc
    import os

    def train():
        ctx = S.Context()
        if name.endswith("images"):
            net = N.resnet20(16)
            g, _ = behind_resize(net, 1536)
        else:
            net = TRAINED[name]()
            g, _ = N.build_graph(net, np.zeros((net.batch,) + tuple(net.in_shape), np.float32))
        p = ctx.create_program(g, net.batch, training=True)
        p.run(2)
        if with_inference:
            q = ctx.create_program(g, net.batch, training=False)
            q.run(1)
            p.run(1)
        return any(op["side"] for op in stub_gpu.plan(p))

    def run(total):
        gc.collect()
        start = stub_gpu.stub.hipstub_used()
        stub_gpu.stub.hipstub_set_memory(total + start)
        stub_gpu.stub.hipstub_peak()
        side = train()
        return stub_gpu.stub.hipstub_peak() - start, side

    train()  # (what the library keeps)
    os.environ["SAGA_HIP_ONE_STREAM"] = "1"
    least, side = run(1 << 38)
    assert not side
    del os.environ["SAGA_HIP_ONE_STREAM"]
    assert run(1 << 38)[1]
    sides = [run(int(least * f))[1] for f in (1, 1.02, 1.1, 1.25, 1.5, 2, 40)]  # (running out of memory ends the process)
    assert sides == sorted(sides) and sides[-1], sides


@on_stub
def test_what_is_recorded_after_the_second_stream_is_given_up():
    """The operations are in another order then: which of their launches may go into a graph is asked again."""
    import os

    os.environ["SAGA_HIP_GRAPH"] = "1"
    net = TRAINED["resnet20"]()
    g, _ = N.build_graph(net, np.zeros((net.batch,) + tuple(net.in_shape), np.float32))
    ctx = S.Context()
    p = ctx.create_program(g, net.batch, training=True)
    p.run(4)
    before = stub_gpu.plan(p)
    assert any(op["side"] for op in before) and any(op["recorded"] for op in before)
    stub_gpu.stub.hipstub_set_memory(stub_gpu.stub.hipstub_used())
    q = ctx.create_program(g, net.batch, training=False)
    stub_gpu.stub.hipstub_set_memory(stub_gpu.stub.hipstub_used() + (1 << 20))
    q.finalize()
    ops = stub_gpu.plan(p)
    assert not any(op["side"] for op in ops) and [op["kind"] for op in ops] != [op["kind"] for op in before]
    stub_gpu.stub.hipstub_set_memory(1 << 38)
    for _ in range(2):
        assert all(op["safe"] for op in stub_gpu.plan(p) if op["recorded"])
        p.run(1)
    assert any(op["recorded"] for op in stub_gpu.plan(p))


@on_stub
def test_late_looks_do_not_end_the_recording():
    """Each has the operations cut into segments anew; their batched tensors are as many as before."""
    import os

    os.environ["SAGA_HIP_GRAPH"] = "1"
    net = N.resnet20(4, dtype=S.FLOAT)
    g, t = N.build_graph(net, np.zeros((4,) + tuple(net.in_shape), np.float32), with_classifier=False)
    ctx = S.Context()
    p = ctx.create_program(g, 4, training=False, batched={t[net.input]: S.PRE, t[net.output]: S.POST})
    p.run(3)
    looks = 0
    for n in net.nodes:
        before = len(stub_gpu.plan(p))
        ctx.resolve(t[n["out"]])
        looks += len(stub_gpu.plan(p)) > before
        p.run(1)
    assert looks > 8
    before = stub_gpu.replays()
    p.run(1)
    assert stub_gpu.replays() > before


@pytest.mark.parametrize("others", [[1, 1], [1, 1, 3], [3, 1, 1]], ids=str)
@on_stub
def test_several_strided_writers_of_a_gradient(others):
    """1x1 convolutions at stride 2 write a quarter of a gradient: those go behind a dense writer, if there is one, and the order
    among themselves is left alone."""
    rng = np.random.default_rng(2)
    draw = lambda *shape: S.Tensor.from_numpy(rng.standard_normal(shape).astype(np.float16), name=f"p{shape}{rng.integers(1 << 40)}")
    g = S.Graph()
    x = g.add_node("conv", {"x": draw(2, 16, 8, 8), "w": draw(16, 16, 3, 3)}, {"size": 3, "activations": 16, "pad": 1}).y()
    ys = [g.add_node("conv", {"x": x, "w": draw(16, 16, r, r)}, {"size": r, "activations": 16, "pad": r // 2, "stride": 2}).y() for r in others]
    y = ys[0]
    for other in ys[1:]:
        y = g.add_node("sum", {"x0": y, "x1": other}).y()
    y = g.add_node("fc", {"x": g.add_node("avgpool", {"x": y}, {"global": True}).y(), "w": draw(16, 10)}, {"outputs": 10}).y()
    g.add_node("catclassifier", {"x": y})
    ctx = S.Context()
    p = ctx.create_program(g, 2, training=True)
    p.finalize()
    ops = stub_gpu.plan(p)
    gradient = [op for op in ops if op["kind"].startswith("convbwddata")]
    filters = [size for op in gradient for _, _, size, name in op["reads"] if name == "w"]
    want = [16 * 16 * r * r * 2 for r in others]
    assert len(filters) == len(others) and sorted(filters) == sorted(want)
    assert filters[0] == max(want)  # the dense one, where there is one, overwrites


@on_stub
def test_small_operations_share_an_edge():
    """An edge between the streams costs the host as much as several launches: weight gradients that are done sooner share one, large
    ones have their own."""

    def edges(net):
        ctx = S.Context()
        g, _ = N.build_graph(net, np.zeros((net.batch,) + tuple(net.in_shape), np.float32))
        p = ctx.create_program(g, net.batch, training=True)
        p.finalize()
        ops = stub_gpu.plan(p)
        assert not stub_gpu.unordered(ops)
        filters = [op for op in ops if op["side"] and op["kind"] == "convbwdfilter"]
        return len({op["fork"] for op in filters} - {-1}), len(filters)

    few, count = edges(N.resnet20(16))
    assert 6 <= few <= 0.7 * count
    all_, count = edges(N.resnet20(8192))
    assert all_ >= 0.9 * count
