"""Training steps with the weight gradients on the side stream against steps on one stream: every kernel is deterministic, so
losses and weights agree bit for bit - with storages that share memory as soon as their last reader is done, and repeatedly."""
import numpy as np
import pytest

from saga_amd import api as S
from saga_amd import networks as N
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
