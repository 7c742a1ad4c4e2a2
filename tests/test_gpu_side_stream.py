"""Training steps with the weight gradients on the side stream against steps on one stream: every kernel is deterministic, so
losses and weights agree bit for bit - with storages that share memory as soon as their last reader is done, and repeatedly."""
import numpy as np
import pytest

from saga_amd import api as S
from saga_amd import networks as N
from tests.test_engine_plan import behind_resize
from tests.test_gpu_graphs import CASES, train

pytestmark = pytest.mark.gpu

MORE = [("resnet50 fp16", lambda: N.resnet50(3, image=72), ["res2_0-conv-1-w", "fc-b"], 32768.0)]


@pytest.mark.parametrize("name,make,params,loss_scale", CASES + MORE, ids=[c[0] for c in CASES + MORE])
def test_side_stream_matches_one_stream(name, make, params, loss_scale, monkeypatch):
    net = make()
    params = [k for k in params if k in net.params] or sorted(net.params)[:4]
    two, w_two = train(net, 12, False, params, loss_scale)
    monkeypatch.setenv("SAGA_HIP_ONE_STREAM", "1")
    one, w_one = train(make(), 12, False, params, loss_scale)
    for i, (a, b) in enumerate(zip(two, one)):
        np.testing.assert_array_equal(a[0], b[0], err_msg=f"{name}: loss after step {i}")
        np.testing.assert_array_equal(a[1], b[1], err_msg=f"{name}: logits after step {i}")
    for k in params:
        np.testing.assert_array_equal(w_two[k], w_one[k], err_msg=f"{name}: weights {k}")


@pytest.mark.parametrize("make,image", [(lambda: N.resnet20(16), 256), (lambda: N.resnet50(3, image=64), 512)], ids=["resnet20", "resnet50"])
def test_large_images_in_front(make, image, monkeypatch):
    """Converted and resized in front of the network: those tensors are large and done with before the first convolution, and the
    filters that the side stream transposes from the start of the step must not be in their memory."""

    def run():
        net, rng = make(), np.random.default_rng(5)
        pixels = rng.integers(0, 256, (net.batch, 3, image, image)).astype(np.uint8)
        g, t = behind_resize(net, image, S.Tensor.from_numpy(pixels, name="pixels"))
        ctx = S.Context()
        p = ctx.create_program(g, net.batch, training=True, learning_rate=1e-3, initial_loss_scale=1024.0)
        p.finalize()
        ctx.resolve(t["labels"]).write(rng.integers(0, net.classes, (net.batch, 1)).astype(np.int32))
        out = [ctx.resolve(t[k]) for k in ("loss", net.output, next(k for k in net.params if net.params[k].ndim == 4))]
        trace = []
        for _ in range(4):
            p.run(2)
            trace.append([v.read().copy() for v in out])
        return trace

    two = run()
    monkeypatch.setenv("SAGA_HIP_ONE_STREAM", "1")
    for i, (a, b) in enumerate(zip(two, run())):
        for x, y in zip(a, b):
            np.testing.assert_array_equal(x, y, err_msg=f"after step {2 * i + 2}")
    assert np.isfinite(two[-1][0]).all() and not np.array_equal(two[0][2], two[-1][2])
