"""Training programs fold relus into the operations in front of them, and their backward into that of a max pooling or product.
Whoever looks at a tensor that went that way still finds its values, and steps are the same to the last bit."""
import ctypes as C

import numpy as np
import pytest
import torch

from saga_amd import api as S
from saga_amd import kernels as K
from saga_amd import networks as N
from tests import stub_gpu
from tests.gpu_util import dev, rnd
from tests.stub_gpu import on_stub

# outputs of the nodes in front of relus, and outputs of relus, whose gradients went away
INPUTS, OUTPUTS = ["c1", "c2", "fc1"], ["relu1", "relu2", "relu3"]


def lenet(batch=6, labels=True, **config):
    net = N.lenet(batch)
    rng = np.random.default_rng(4)
    x = rng.standard_normal((batch,) + tuple(net.in_shape)).astype(np.float32)
    g, t = N.build_graph(net, x)
    relus = [n for n in net.nodes if n["type"] == "relu"]
    assert len(relus) == 3
    for name, out, n in zip(INPUTS, OUTPUTS, relus):
        t[name], t[out] = t[n["in"]["x"]], t[n["out"]]
    ctx = S.Context()
    p = ctx.create_program(g, batch, training=True, **config)
    if labels:
        ctx.resolve(t["labels"]).write(rng.integers(0, 10, (batch, 1)).astype(np.int32))
    return net, ctx, p, t


def kinds(p):
    return [op["kind"] for op in stub_gpu.plan(p)]


@on_stub
def test_relus_are_folded_away():
    _, ctx, p, t = lenet(labels=False)
    p.finalize()
    assert not [k for k in kinds(p) if k.startswith("act")]
    assert len([k for k in kinds(p) if k == "poolbwd"]) == 2
    before = stub_gpu.plan(p)
    for name in INPUTS:
        ctx.resolve(t[name])
    for name in OUTPUTS:
        ctx.resolve(t[name].grad())
    after = stub_gpu.plan(p)
    assert [op["kind"] for op in after] == [op["kind"] for op in before]
    assert all(address for op in after for _, address, *_ in op["writes"])  # (nothing is allocated while launches are recorded)
    assert sum(len(op["writes"]) for op in after) == sum(len(op["writes"]) for op in before) + 6
    p.run(1)
    assert stub_gpu.unordered(after) == [] and stub_gpu.overlapping(after) == []


@on_stub
def test_relus_that_somebody_sees_are_not():
    _, ctx, p, t = lenet(labels=False)
    ctx.resolve(t["c1"])
    ctx.resolve(t["relu2"].grad())
    p.finalize()
    assert sorted(k for k in kinds(p) if k.startswith("act")) == ["actbwd", "actfwd"]
    for config in (dict(disable_op_fusing=True), dict(anomaly_detect=True)):
        _, _, q, _ = lenet(labels=False, **config)
        q.finalize()
        assert len([k for k in kinds(q) if k.startswith("act")]) == 6


@pytest.mark.gpu
@pytest.mark.parametrize("graphs", [False, True])
def test_steps_are_the_same(graphs, monkeypatch):
    if graphs:
        monkeypatch.setenv("SAGA_HIP_GRAPH", "1")
    names = INPUTS + OUTPUTS
    state = {}
    for fused in (False, True):
        net, ctx, p, t = lenet(disable_op_fusing=not fused)
        loss = ctx.resolve(t["loss"])
        p.finalize()
        p.run(2)
        seen = {}
        for name in names:  # one after the other: what was folded with the last is undone between steps
            d = ctx.resolve(t[name] if name in INPUTS else t[name].grad())
            p.run(1)
            seen[name] = d.read().copy()
        p.run(3)
        seen.update({k: ctx.resolve(t[k]).read().copy() for k in net.params}, loss=loss.read().copy())
        state[fused] = seen
    for k, v in state[False].items():
        assert np.abs(v).max() > 0 and np.array_equal(v, state[True][k]), k


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("size,H,W", [(2, 8, 8), (2, 9, 11), (3, 9, 9), (3, 11, 10), (2, 2, 2)])
def test_pooling_and_relu_backward(size, H, W, dtype):
    rng = np.random.default_rng(H + W)
    P, Q = H // size, W // size
    x = np.maximum(rnd(rng, 3, 5, H, W, dtype=dtype), 0)  # windows of nothing but zeros among them
    x[1, 2, :size, :size] = 0
    x[2, 1, 0, 0] = np.nan
    y = np.zeros((3, 5, P, Q), np.float32)
    dy = rnd(rng, 3, 5, P, Q, dtype=dtype)
    dy[0, 0, 0, 0] = np.inf
    xd, yd, gd = dev(x, dtype), dev(y, dtype), dev(dy, dtype)
    L, V = K.lib(), lambda a: C.byref(K.view(a))
    K.check(L.saga_hip_pool_fwd(K.POOL_MAX, V(xd), V(yd), None, size, 0, size, K.stream_ptr()))
    between, want, got = (torch.full_like(xd, 7.0) for _ in range(3))
    K.check(L.saga_hip_pool_bwd(K.POOL_MAX, V(xd), V(yd), V(gd), V(between), size, 0, size, 0.0, K.stream_ptr()))
    K.check(L.saga_hip_act_bwd(0, 0.0, V(xd), V(xd), V(between), V(want), 0.0, K.stream_ptr()))
    assert L.saga_hip_maxpool_bwd_relu_ok(V(xd), V(yd), V(gd), V(got), size, 0, size)
    K.check(L.saga_hip_maxpool_bwd_relu(V(xd), V(yd), V(gd), V(got), size, 0, size, K.stream_ptr()))
    assert torch.equal(torch.nan_to_num(got, nan=99.0), torch.nan_to_num(want, nan=99.0))
    last = dev(x, dtype, "nhwc")
    assert not L.saga_hip_maxpool_bwd_relu_ok(V(last), V(yd), V(gd), V(got), size, 0, size)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("M,N_,Kd,tA,tB", [(6, 1024, 10, 0, 1), (33, 65, 70, 0, 0), (64, 500, 512, 0, 1), (7, 3, 5, 1, 0)])
def test_product_and_relu_backward(M, N_, Kd, tA, tB, dtype):
    rng = np.random.default_rng(M)
    code = K.HALF if dtype == torch.float16 else K.FLOAT
    A, B = rnd(rng, M, Kd, dtype=dtype), rnd(rng, Kd, N_, dtype=dtype)
    Ad, Bd = dev(A.T if tA else A, dtype), dev(B.T if tB else B, dtype)
    y = np.maximum(rnd(rng, M, N_, dtype=dtype), 0)
    y[0, 0] = np.nan
    yd = dev(y, dtype)
    between, want, got = (torch.full((M, N_), 7.0, device="cuda", dtype=dtype) for _ in range(3))
    L, V = K.lib(), lambda a: C.byref(K.view(a.view(M, N_, 1, 1)))
    assert L.saga_hip_gemm_relu_bwd_ok(M, N_, Kd, code)
    K.check(L.saga_hip_gemm(tA, tB, M, N_, Kd, 1.0, K.ptr(Ad), Ad.shape[1], K.ptr(Bd), Bd.shape[1], 0.0, K.ptr(between), N_, code,
                            K.stream_ptr()))
    K.check(L.saga_hip_act_bwd(0, 0.0, V(yd), V(yd), V(between), V(want), 0.0, K.stream_ptr()))
    K.check(L.saga_hip_gemm_relu_bwd(tA, tB, M, N_, Kd, 1.0, K.ptr(Ad), Ad.shape[1], K.ptr(Bd), Bd.shape[1], K.ptr(got), N_, code,
                                     K.ptr(yd), K.stream_ptr()))
    assert torch.equal(got, want)
    assert not L.saga_hip_gemm_relu_bwd_ok(4096, 4096, 64, code)
