"""The work that users of this framework have it do, as cases that can be timed and compared.

Two kinds of pass.  A network pass goes through Graph -> Context -> Program (saga_amd.api): one inference batch or
one training step (forward, backward, Adam) of a network of saga_amd.networks.  A layer pass goes through the C ABI
(saga_amd.kernels): one convolution layer forward, backward data and backward filter.

A case is a dict of plain values:
    net    "resnet50", "resnet20", "lenet", "unet", or "conv" for a layer pass
    mode   "infer" or "train" (network passes)
    dtype  "f16" (channels-last, matrix cores in fp16) or "f32" (channels-first)
    batch, image    samples per pass, pixels per side
    feed   how the batch gets to the GPU: "device" (it is there already), "write" (Tensor.write into the program's
           input before the pass, the way a request is served) or "batched" (a batched tensor: the program uploads
           the host's back buffers itself, the way a training loop is fed)
    c, k, r, stride  input and output channels, filter side and stride (layer passes; pad is r // 2)
"""
import copy
import functools
import math

import numpy as np
import torch

from saga_amd import api as S
from saga_amd import kernels as K
from saga_amd import networks as N

_DTYPE = {"f16": S.HALF, "f32": S.FLOAT}
_TORCH = {"f16": torch.float16, "f32": torch.float32}
_SIZE = {"f16": 2, "f32": 4}


def _net(net, mode, dtype, batch, image, feed):
    return {"net": net, "mode": mode, "dtype": dtype, "batch": batch, "image": image, "feed": feed}


def _conv(dtype, batch, image, c, k, r, stride):
    return {"net": "conv", "dtype": dtype, "batch": batch, "image": image, "c": c, "k": k, "r": r, "stride": stride}


def listed():
    cases = {
        # one image at a time behind a service: the request comes from the host and its scores go back
        "resnet50 serve 1": _net("resnet50", "infer", "f16", 1, 224, "write"),
        # a model as ONNX files hold it (fp32, channels-first) answering small batches
        "resnet50 serve 8 f32": _net("resnet50", "infer", "f32", 8, 224, "write"),
        # offline inference, the benchmark's batch
        "resnet50 infer 256": _net("resnet50", "infer", "f16", 256, 224, "device"),
        # the benchmark's training step
        "resnet50 train 256": _net("resnet50", "train", "f16", 256, 224, "device"),
        # fine-tuning at a resolution of one's own, on the short batch that a data set leaves over
        "resnet50 train 23 at 193": _net("resnet50", "train", "f16", 23, 193, "device"),
        # the digits classifier: scoring a batch, and the training loop that made it
        "lenet infer 64": _net("lenet", "infer", "f32", 64, 28, "write"),
        "lenet train 64": _net("lenet", "train", "f32", 64, 28, "batched"),
        # training on small images: many layers of little work each
        "resnet20 train 128": _net("resnet20", "train", "f16", 128, 32, "batched"),
        # segmentation: training on crops, and one whole image with the per-pixel softmax on top
        "unet train 16": _net("unet", "train", "f16", 16, 256, "device"),
        "unet segment 1": _net("unet", "infer", "f16", 1, 336, "write"),
        # the single-layer microbenchmark of bench.py, in both precisions
        "conv layer f16": _conv("f16", 256, 56, 64, 64, 3, 1),
        "conv layer f32": _conv("f32", 256, 56, 64, 64, 3, 1),
    }
    return [dict(c, name=name) for name, c in cases.items()]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["resnet50", "resnet50", "resnet20", "lenet", "unet", "conv", "conv"])
    mode = rng.choice(["infer", "train"])
    if kind == "resnet50":
        image = rng.randint(128, 256)
        if mode == "train":  # batch norm in training mode wants more than a handful of samples
            return _net(kind, mode, "f16", _log(rng, 16, 96), image, rng.choice(["device", "batched"]))
        dtype = rng.choice(["f16", "f16", "f32"])
        return _net(kind, mode, dtype, _log(rng, 1, 128 if dtype == "f16" else 32), image, rng.choice(["device", "write"]))
    if kind == "resnet20":
        return _net(kind, mode, rng.choice(["f16", "f32"]), _log(rng, 16, 512), 32, "batched" if mode == "train" else "write")
    if kind == "lenet":
        return _net(kind, mode, "f32", _log(rng, 4, 512), 28, "batched" if mode == "train" else "write")
    if kind == "unet":
        image = 16 * rng.randint(8, 22)
        most = max(1, 16 * 256 * 256 // (image * image))
        batch = rng.randint(2, max(2, most // 2)) if mode == "train" else _log(rng, 1, most)
        return _net(kind, mode, "f16", batch, image, "device" if mode == "train" else "write")
    dtype = rng.choice(["f16", "f16", "f32"])
    image, r, stride = _log(rng, 7, 112), rng.choice([1, 3, 3, 5]), rng.choice([1, 1, 2])
    c, k = _log(rng, 8, 512), _log(rng, 8, 512)
    if rng.random() < 0.5:  # most layers have channels in eights
        c, k = -(-c // 8) * 8, -(-k // 8) * 8
    most = 59e9 / (2.0 * c * k * r * r * (image / stride) ** 2)  # the listed layers' operations
    fits = 6e8 / (max(c, k) * image * image)  # and no more than their memory several times
    return _conv(dtype, _log(rng, 1, max(1, min(256, most, fits))), image, c, k, r, stride)


@functools.lru_cache(maxsize=16)
def _described(kind, mode, dtype, image):
    """The network with its seeded initial weights, for one sample."""
    if kind == "lenet":
        return N.lenet(1)
    if kind == "resnet20":
        return N.resnet20(1, dtype=_DTYPE[dtype])
    if kind == "resnet50":
        return N.resnet50(1, dtype=_DTYPE[dtype], image=image)
    net = N.unet(1, dtype=_DTYPE[dtype], image=image, softmax=mode == "infer")
    if mode == "train":  # a scalar loss: the class scores of all pixels pooled into one set of scores
        b = N.Builder(net, 99)
        b.shape[net.output] = (net.classes, image, image)
        net.output = b.fc(b.pool("avgpool", net.output, global_=True), "cls", net.classes)
    return net


def _network(case):
    net = copy.copy(_described(case["net"], case["mode"], case["dtype"], case["image"]))
    net.batch = net.rows = case["batch"]
    return net


class _OnDevice(dict):
    """What a training step leaves in the program: weights, batch-norm parameters and running statistics.  They stay on
    the device, as in a training loop, and an entry is fetched when it is looked up."""

    def __init__(self, ctx, tensors, groups):
        super().__init__(dict.fromkeys(groups))
        self._fetch = lambda key: np.concatenate([ctx.resolve(tensors[n]).read().ravel() for n in groups[key]])

    def __getitem__(self, key):
        return self._fetch(key)


def _groups(net):
    norm = [n for n in net.params if n.endswith("-s")]
    norm += [n[:-2] + "-b" for n in norm]
    running = [n for n in net.params if n.endswith(("-m", "-v"))]
    weights = [n for n in net.params if n not in norm and n not in running]
    return {k: v for k, v in (("weights", weights), ("norm", norm), ("running", running)) if v}


def _prepare_network(case, gen, seed):
    net = _network(case)
    shape = (net.batch,) + tuple(net.in_shape)
    if net.name == "lenet":  # grey values
        x = torch.rand(shape, device="cuda", generator=gen)
    else:  # colours after the usual normalisation
        x = torch.randn(shape, device="cuda", generator=gen)
    x = x.to(_TORCH[case["dtype"]]).cpu().numpy()
    train, feed = case["mode"] == "train", case["feed"]
    labels = np.random.default_rng(seed).integers(0, net.classes, (net.batch, 1)).astype(np.int32)
    ctx = S.Context()
    graph, t = N.build_graph(net, x, with_classifier=train)
    batched = None
    if feed == "batched":
        batched = {t[net.input]: S.PRE}
        if train:
            batched[t["labels"]] = S.PRE
    program = ctx.create_program(graph, net.batch, training=train, batched=batched,
                                 initial_loss_scale=4096.0 if net.name == "unet" else 1024.0)
    state = {"program": program, "graph": graph, "tensors": t, "x": x, "labels": labels, "feed": feed,
             "input": ctx.resolve(t[net.input])}
    if train:
        state["target"], state["result"] = ctx.resolve(t["labels"]), ctx.resolve(t["loss"])
        state["trained"] = _OnDevice(ctx, t, _groups(net))
        if feed == "device":
            state["target"].write(labels)
    else:
        state["result"] = ctx.resolve(t[getattr(net, "softmax", None) or net.output])
    program.finalize()
    return state


def _run_network(state):
    if state["feed"] != "device":
        state["input"].write(state["x"])
        if "target" in state:
            state["target"].write(state["labels"])
    state["program"].run(1)
    out = {"result": state["result"].read()}
    if "trained" in state:
        out["trained"] = state["trained"]
    return out


def _conv_shapes(case):
    n, c, k, r, h = case["batch"], case["c"], case["k"], case["r"], case["image"]
    p = 1 + (h + 2 * (r // 2) - r) // case["stride"]
    return (n, c, h, h), (k, c, r, r), (n, k, p, p)


def _prepare_conv(case, gen):
    xs, ws, ys = _conv_shapes(case)
    dt = _TORCH[case["dtype"]]
    fmt = torch.channels_last if case["dtype"] == "f16" else torch.contiguous_format

    def make(shape, scale=1.0):
        a = torch.randn(shape, device="cuda", generator=gen).mul_(scale)
        return a.to(dt).contiguous(memory_format=fmt)

    def empty(shape):
        return torch.empty(shape, device="cuda", dtype=dt, memory_format=fmt)

    # the loss gradient of a batch is small; dw adds up batch * pixels of these
    dy = make(ys, 1.0 / math.sqrt(ys[0] * ys[2] * ys[3]))
    return {"x": make(xs), "w": make(ws, math.sqrt(2.0 / (ws[1] * ws[2] * ws[3]))), "dy": dy, "y": empty(ys),
            "dx": empty(xs), "dw": empty(ws), "pad": case["r"] // 2, "stride": case["stride"]}


def _run_conv(s):
    K.conv2d(K.CONV_FWD, s["x"], s["w"], s["y"], s["pad"], s["stride"])
    K.conv2d(K.CONV_BWD_DATA, s["dy"], s["w"], s["dx"], s["pad"], s["stride"])
    K.conv2d(K.CONV_BWD_FILTER, s["x"], s["dy"], s["dw"], s["pad"], s["stride"])
    return {"y": s["y"], "dx": s["dx"], "dw": s["dw"]}


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return _prepare_conv(case, gen) if case["net"] == "conv" else _prepare_network(case, gen, seed)


def run(state):
    return _run_network(state) if "program" in state else _run_conv(state)


def work(case):
    size = _SIZE[case["dtype"]]
    if case["net"] == "conv":
        xs, ws, ys = _conv_shapes(case)
        # x, w, dy read and y, dx, dw written
        return {"bytes": 2 * size * (math.prod(xs) + math.prod(ws) + math.prod(ys)), "flops": 3 * 2.0 * math.prod(ys) * math.prod(ws[1:])}
    net = _network(case)
    params = sum(a.size for a in net.params.values())
    moved = case["batch"] * math.prod(net.in_shape) * size
    if case["mode"] == "infer":
        pixels = case["image"] ** 2 if case["net"] == "unet" else 1
        return {"bytes": moved + params * size + case["batch"] * net.classes * pixels * size, "flops": net.flops_fwd * case["batch"]}
    # forward, backward data and backward filter; the first convolution needs no backward data
    a = net.nodes[0]["attrs"]
    c, h, _ = net.in_shape
    side = 1 + (h + 2 * a["pad"] - a["size"]) // a["stride"]
    first = 2.0 * side * side * a["activations"] * c * a["size"] ** 2
    # Adam reads and writes each weight, both moments and, in fp16, the fp32 master weight
    return {"bytes": moved + params * (28 if size == 2 else 24) + case["batch"] * 4, "flops": (3 * net.flops_fwd - first) * case["batch"]}


def tolerance(case):
    if case["net"] == "conv":  # fp32 sums in another order; results rounded to fp16
        return {"rel": 1e-3, "max": 1e-2} if case["dtype"] == "f16" else {"rel": 1e-5, "max": 1e-3}
    if case["mode"] == "infer":  # up to 53 layers, each stored in fp16 / summed in fp32
        return {"rel": 1e-2, "max": 0.2} if case["dtype"] == "f16" else {"rel": 2e-5, "max": 1e-3}
    # Adam's first step moves a weight by the learning rate in the direction of its gradient's sign, so a gradient within
    # rounding of zero moves its weight the other way: 1e-4 either way beside weights of 1e-2
    return {"rel": 2e-2, "max": 0.2} if case["dtype"] == "f16" else {"rel": 5e-5, "max": 5e-2}
