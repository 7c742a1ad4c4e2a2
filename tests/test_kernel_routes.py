"""Which kernels the library's entry points launch, and what they refuse, without a GPU (over the stub runtime)."""
import ctypes as C
import re

import pytest

from saga_amd import kernels as K
from tests import stub_gpu
from tests.stub_gpu import on_stub


def image(address, n, c, h, w, pitch=None, dtype=K.HALF):
    """Channels-last; the address is never read."""
    v = K.TensorView()
    p = pitch or c
    v.ptr, v.dtype = address, dtype
    v.dims[:], v.strides[:] = [n, c, h, w], [h * w * p, 1, w * p, p]
    return v


X, Y, W, ROOM = 1 << 20, 1 << 30, 1 << 31, 1 << 32


def gradient(kind, x, w, y, room):
    """Return code of a backward pass, and whether the direct kernel and a matrix-core kernel ran."""
    L, p = K.lib(), K.ConvParams(1, 1, 1, 1)
    before = [stub_gpu.launches(k) for k in ("direct_", "conv_bwd_filter_dma", "stream_f16", "conv_gather")]
    ptr = ROOM if room else None
    if kind == K.CONV_BWD_DATA:
        rc = L.saga_hip_conv2d_bwd_data(C.byref(y), C.byref(w), C.byref(x), C.byref(p), 1.0, 0.0, ptr, room, None)
    else:
        rc = L.saga_hip_conv2d_bwd_filter(C.byref(x), C.byref(y), C.byref(w), C.byref(p), 1.0, 0.0, ptr, room, None)
    ran = [stub_gpu.launches(k) - b for k, b in zip(("direct_", "conv_bwd_filter_dma", "stream_f16", "conv_gather"), before)]
    return rc, ran[0] > 0, any(ran[1:])


@pytest.mark.parametrize("k,pitch", [(21, 21), (24, 28), (24, 24)])
@pytest.mark.parametrize("kind", [K.CONV_BWD_DATA, K.CONV_BWD_FILTER])
@on_stub
def test_fp16_gradients_without_room_for_a_padded_copy(kind, k, pitch):
    """Output channels or a pitch that are no multiple of eight: the copy needs workspace, a call without any is still served."""
    x, w, y = image(X, 4, 16, 30, 30), image(W, k, 16, 3, 3), image(Y, 4, k, 30, 30, pitch)
    need = K.lib().saga_hip_conv2d_workspace_size(kind, C.byref(x), C.byref(w), C.byref(y), C.byref(K.ConvParams(1, 1, 1, 1)))
    assert gradient(kind, x, w, y, need) == (0, False, True)
    odd = pitch % 8 != 0
    for room in (0, 1024, 4 * 30 * 30 * 24 * 2):  # the last holds the copy alone
        if odd:
            assert gradient(kind, x, w, y, room) == (0, True, False), room
    if not odd:  # (such tensors have always needed theirs)
        assert gradient(kind, x, w, y, 0)[0] == -4


@on_stub
def test_padded_copies_by_their_size():
    """A vector to a thread in small ones, both operands' in one launch."""
    L, p = K.lib(), K.ConvParams(0, 1, 1, 1)
    for n, c, k, image_size, want in ((5, 64, 122, 13, [1, 53]), (5, 65, 122, 13, [1, 83]), (64, 64, 122, 60, [4, 3600])):
        x, w, y = image(X, n, c, image_size, image_size), image(W, k, c, 1, 1), image(Y, n, k, image_size, image_size)
        stub_gpu.launched()
        assert L.saga_hip_conv2d_bwd_filter(C.byref(x), C.byref(y), C.byref(w), C.byref(p), 1.0, 0.0, ROOM, 1 << 30, None) == 0
        pads = [(args, blocks) for name, args, blocks, _ in stub_gpu.launched() if name == "pad_channels"]
        assert len(pads) == 1 and pads[0][0] == tuple(want[:1]) and pads[0][1] == want[1]


@pytest.mark.parametrize("c,k,r", [(16, 64, 3), (8, 64, 5), (7, 13, 3)])
@on_stub
def test_fp32_filter_gradients_with_fewer_partials(c, k, r):
    """The reduction is split as often as the workspace allows, down to once."""
    p = K.ConvParams(r // 2, 1, 1, 1)
    x, w, y = (image(a, *d, dtype=K.FLOAT) for a, d in ((X, (8, c, 28, 28)), (W, (k, c, r, r)), (Y, (8, k, 28, 28))))
    L = K.lib()
    need = L.saga_hip_conv2d_workspace_size(K.CONV_BWD_FILTER, C.byref(x), C.byref(w), C.byref(y), C.byref(p))
    once = 4 * k * c * r * r
    table = 64 * c * r * r + 1024  # more than the general kernel's table of offsets takes
    assert need > 4 * (once + table)
    for room, want in ((need, 0), (need // 2, 0), (once + table, 0), (once - 4, -4), (0, -4)):
        rc = L.saga_hip_conv2d_bwd_filter(C.byref(x), C.byref(y), C.byref(w), C.byref(p), 1.0, 0.0, ROOM if room else None, room, None)
        assert rc == want, (room, rc)


@pytest.mark.parametrize("dtype", [K.HALF, K.FLOAT])
@on_stub
def test_norms_of_planes(dtype):
    """Channels that a block holds take one launch, others two; inference goes through the values in their order in memory."""
    L = K.lib()
    channel = [ROOM + (i << 20) for i in range(8)]
    vector = 8 if dtype == K.HALF else 4

    def ran(n, c, h, w):
        t = [image(a, n, c, h, w, dtype=dtype) for a in (X, Y, W)]
        for v in t:
            v.strides[:] = [c * h * w, h * w, w, 1]
        x, y, dy = (C.byref(v) for v in t)
        stub_gpu.launched()
        s, b, m, v, mean, std, ds, db = channel
        ws = 64 * ROOM, 1 << 30
        assert L.saga_hip_bn_train_fwd(x, None, y, s, b, m, v, mean, std, 1e-5, 0.1, K.BN_RELU, *ws, None) == 0
        assert L.saga_hip_bn_bwd(x, y, dy, dy, None, s, mean, std, ds, db, 0.0, 0.0, 0.0, K.BN_RELU, *ws, None) == 0
        train = [name for name, *_ in stub_gpu.launched()]
        assert L.saga_hip_bn_infer(x, None, y, s, b, m, v, 1e-5, K.BN_RELU, None) == 0
        return train, [name for name, *_ in stub_gpu.launched()]

    one, two = ["bn_apply_cf", "bn_bwd_apply_cf"], ["bn_stats_cf", "bn_apply_cf", "bn_bwd_stats_cf", "bn_bwd_apply_cf"]
    assert ran(1, 512, 7, 7) == (one, ["bn_infer_cf"])
    assert ran(8, 2048, 7, 7) == (one, ["bn_infer_cf"])
    assert ran(512, 64, 2, 2) == (one if dtype == K.FLOAT else two, ["bn_infer_cf"])
    assert ran(1024 // 64, 4, 8, 8 * vector) == (one, ["bn_infer_cf"])
    assert ran(1024 // 64 + 1, 4, 8, 8 * vector) == (two, ["bn_infer_cf"])
    assert ran(512, 512, 7, 7) == (two, ["bn_apply_cf" if dtype == K.HALF else "bn_infer_cf"])


@on_stub
def test_biases_that_are_no_vector_are_refused():
    """Elements at no constant distance; a constant one other than 1 goes to a pass of its own."""
    x, w, y, p = image(X, 2, 16, 9, 9), image(W, 16, 16, 3, 3), image(Y, 2, 16, 9, 9), K.ConvParams(1, 1, 1, 1)
    L = K.lib()
    n = L.saga_hip_conv2d_workspace_size(K.CONV_FWD, C.byref(x), C.byref(w), C.byref(y), C.byref(p))
    for dims, strides, want, passes in (([1, 16, 1, 1], [16, 1, 1, 1], 0, 0), ([16, 1, 1, 1], [1, 1, 1, 1], 0, 0),
                                        ([4, 1, 4, 1], [4, 9, 1, 9], 0, 0), ([1, 16, 1, 1], [1, 3, 1, 1], 0, 1),
                                        ([4, 1, 4, 1], [12, 9, 3, 9], 0, 1), ([4, 4, 1, 1], [5, 1, 1, 1], -3, 0),
                                        ([1, 15, 1, 1], [1, 1, 1, 1], -2, 0)):
        b = image(1 << 33, 1, 16, 1, 1)
        b.dims[:], b.strides[:] = dims, strides
        before = stub_gpu.launches("bias_add")
        e = K.ConvExtras(bias=C.pointer(b))
        rc = L.saga_hip_conv2d_fwd_ex(C.byref(x), C.byref(w), C.byref(y), C.byref(p), 0.0, C.byref(e), ROOM, n, None)
        assert (rc, stub_gpu.launches("bias_add") - before) == (want, passes), (dims, strides)
        assert L.saga_hip_bias_add(C.byref(y), C.byref(b), None) == want


def convolution(kind, shape, dtype, bias=False, room=1.0):
    """The launches of a convolution of dense tensors (forward: also with a bias), and the pixels of its classes and its columns.
    room: bytes of workspace, or (a float) a share of what the query asks for."""
    n, c, h, w, k, r, stride, pad = shape
    p, q = 1 + (h + 2 * pad - r) // stride, 1 + (w + 2 * pad - r) // stride
    x, f, y = (image(a, *d, dtype=dtype) for a, d in ((X, (n, c, h, w)), (W << 2, (k, c, r, r)), (Y << 3, (n, k, p, q))))
    if dtype == K.FLOAT:  # channels-first
        for v in (x, f, y):
            d = v.dims
            v.strides[:] = [d[1] * d[2] * d[3], d[2] * d[3], d[3], 1]
    L, cp = K.lib(), K.ConvParams(pad, stride, 1, 1)
    if isinstance(room, float):
        room = int(room * L.saga_hip_conv2d_workspace_size(kind, C.byref(x), C.byref(f), C.byref(y), C.byref(cp)))
    b = image(1 << 35, 1, k if kind == K.CONV_FWD else c, 1, 1, dtype=dtype)
    stub_gpu.launched()
    if kind == K.CONV_FWD:
        e = K.ConvExtras(bias=C.pointer(b)) if bias else K.ConvExtras()
        rc = L.saga_hip_conv2d_fwd_ex(C.byref(x), C.byref(f), C.byref(y), C.byref(cp), 0.0, C.byref(e), 1 << 36, room, None)
    else:
        rc = L.saga_hip_conv2d_bwd_data_bias(C.byref(y), C.byref(f), None, C.byref(b) if bias else None, C.byref(x), C.byref(cp), 0.0,
                                             1 << 36, room, None)
    assert rc == 0
    classes = [n * p * q] if kind == K.CONV_FWD else [n * -(-(h - a) // stride) * -(-(w - b) // stride) for a in range(stride) for b in range(stride)]
    return stub_gpu.launched(), classes, k if kind == K.CONV_FWD else c


def small_grid_tile(launches, classes, columns):
    """What tests/test_gpu_conv_small_grids.py calls it."""
    split = {(1, 4): "four along the pixels", (2, 2): "two and two", (4, 1): "four along the reduction", (8, 1): "eight along the reduction"}
    for name, t, blocks, threads in launches:
        if name == "stream_f16_k":
            tm, tn = t[:2]
            for (ks, wm), text in split.items():
                if threads == 64 * ks * wm and blocks == sum(-(-m // (16 * tm * wm)) for m in classes) * -(-columns // (16 * tn)):
                    return f"{16 * tm}x{16 * tn}, {text}"
    shared = any(name == "split_reduce" for name, *_ in launches)
    (tile,) = [t for name, t, *_ in launches if name == "conv_gather_gemm_dma"]
    return f"{'shared ' if shared else ''}{tile[0]}x{tile[1]} tiles"


@on_stub
def test_fp16_small_grid_shapes_are_what_their_names_say():
    from tests.test_gpu_conv_small_grids import SHAPES

    seen = set()
    for name, shape in SHAPES.items():
        text = re.sub(r" \([^)]*\)", "", name).replace(", some that no tap reaches,", "")
        forward, _, backward = text.partition("; backward ")
        if forward.startswith("backward "):
            forward, backward = None, forward[len("backward "):]
        for kind, want in ((K.CONV_FWD, forward), (K.CONV_BWD_DATA, backward or forward)):
            if want is None:
                continue
            launches, classes, columns = convolution(kind, shape, K.HALF)
            assert want.startswith("classes of ") == (len(classes) > 1), name
            want = want.replace("classes of ", "")
            got = small_grid_tile(launches, classes, columns)
            assert got == want, (name, kind, got)
            seen.add((kind, len(classes) > 1, got))
    small = ["16x16, four along the pixels", "16x16, four along the reduction", "32x32, two and two", "32x32, four along the reduction",
             "64x32, two and two", "64x32, eight along the reduction", "64x64, two and two", "64x64, four along the reduction"]
    for kind in (K.CONV_FWD, K.CONV_BWD_DATA):
        for tile in small + ["shared 256x128 tiles", "shared 256x64 tiles"]:
            assert (kind, False, tile) in seen, (kind, tile)
    assert (K.CONV_BWD_DATA, True, "shared 256x128 tiles") in seen


# tile rows and columns in 32s, wavefronts along the reduction and along the pixels
F32_TILES = {(2, 8, 255, 257, 65, 1, 1, 0): (2, 2, 1, 4), (1, 1032, 79, 80, 200, 1, 1, 0): (2, 2, 4, 1), (1, 392, 90, 92, 40, 1, 1, 0): (2, 1, 4, 1),
             (1, 16, 311, 317, 7, 1, 1, 0): (2, 1, 1, 4), (3, 64, 9, 7, 31, 1, 1, 0): (1, 1, 1, 4), (1, 24, 180, 183, 72, 3, 1, 1): (2, 2, 1, 4),
             (1, 24, 311, 317, 24, 3, 1, 1): (2, 1, 1, 4), (1, 40, 157, 158, 64, 3, 1, 1): (1, 1, 1, 4), (1, 16, 141, 142, 64, 3, 1, 1): (1, 1, 2, 2),
             (1, 128, 150, 161, 64, 3, 1, 1): (1, 1, 4, 1), (1, 512, 3, 5, 33, 3, 1, 1): (1, 1, 16, 1)}


@on_stub
def test_fp32_shapes_are_what_their_comments_say():
    from tests.test_gpu_stream_f32 import CONVS, LDS

    assert set(F32_TILES) <= set(CONVS)
    for shape, (tm, tn, ks, wm) in F32_TILES.items():
        launches, (pixels,), columns = convolution(K.CONV_FWD, shape, K.FLOAT)
        (tile,) = [x for x in launches if x[0] == "stream_f32_k"]
        assert tile[1][2:4] == (tm, tn) and tile[3] == 64 * ks * wm, (shape, tile)
        assert tile[2] == -(-pixels // (32 * tm * wm)) * -(-columns // (32 * tn)), (shape, tile)
        assert (tile[1][1] == 3) == any(x[0] == "stream_pack_call" for x in launches) == (shape[5] > 1)
    seen = {(kind, name, tile[:2] if "uniform" in name else ()) for shape in LDS for kind in (K.CONV_FWD, K.CONV_BWD_DATA)
            for name, tile, *_ in convolution(kind, shape, K.FLOAT)[0]}
    for kind in (K.CONV_FWD, K.CONV_BWD_DATA):
        assert {(kind, "conv_f32_gather_uniform", (128, 128)), (kind, "conv_f32_gather_uniform", (128, 64)), (kind, "conv_f32_gather", ())} <= seen


# as above; None: tiles in LDS
GEMM_TILES = {(640, 2048, 20): (1, 1, 1, 4), (2890, 3010, 21): (2, 2, 1, 4), (1300, 1290, 1030): (2, 2, 4, 1), (1000, 3100, 20): (2, 1, 1, 4),
              (520, 1060, 390): (2, 1, 4, 1), (640, 1030, 9): None}


@pytest.mark.parametrize("tA,tB", [(0, 0), (0, 1), (1, 0), (1, 1)])
@on_stub
def test_fp32_products_are_what_their_comments_say(tA, tB):
    for (m, n, k), want in GEMM_TILES.items():
        stub_gpu.launched()
        assert K.lib().saga_hip_gemm(tA, tB, m, n, k, 1.0, X, m if tA else k, Y, k if tB else n, 0.0, ROOM, n, K.FLOAT, None) == 0
        ((name, tile, blocks, threads),) = stub_gpu.launched()
        if want is None:
            assert name == "gemm_mfma_f32"
        else:
            tm, tn, ks, wm = want
            got = name, tile[2:4], threads, blocks
            assert got == ("stream_f32_k", (tm, tn), 64 * ks * wm, -(-n // (32 * tm * wm)) * -(-m // (32 * tn))), (m, n, k)


BIAS_KERNELS = {"small grid": "stream_f16_k", "larger tile of a small grid": "stream_f16_k", "shared tiles": "split_reduce",
                "tiles": "conv_gather_gemm_dma", "rows": "conv_rows64", "thin": "conv_thin_rows", "stream": "stream_f32_k", "table": "stream_f32_k"}


@on_stub
def test_fused_bias_shapes_are_what_their_names_say():
    import torch

    from tests.test_gpu_fused_bias import CONVS, TRANSPOSED

    for table, kind in ((CONVS, K.CONV_FWD), (TRANSPOSED, K.CONV_BWD_DATA)):
        for name, (dtype, *shape) in table.items():
            launches = [x[0] for x in convolution(kind, shape[:8], K.HALF if dtype == torch.float16 else K.FLOAT, bias=True)[0]]
            what = max((k for k in BIAS_KERNELS if k in name), key=len, default=None)
            if what == "tiles" and dtype == torch.float32:
                assert any(x.startswith("conv_f32_gather") for x in launches), (name, launches)
            elif what:
                assert any(x.startswith(BIAS_KERNELS[what]) for x in launches), (name, launches)
                assert ("split_reduce" in launches) == (what == "shared tiles"), (name, launches)


# a forward pass or backward data, a workspace in bytes or a share of what is asked for: the kernel, how it reads the filter (fp32 from
# memory: 0 and 1 in place, 2 through a table, 3 packed)
F32_ROUTES = [
    # 1x1 over many pixels: windows where there is room to pack the filter, and otherwise in place as ever
    ((4, 256, 128, 128, 256, 1, 1, 0), K.CONV_FWD, 1.0, "stream_f32_k_window", None),
    ((4, 256, 128, 128, 256, 1, 1, 0), K.CONV_FWD, 0, "stream_f32_k", 0),
    ((4, 256, 128, 128, 256, 1, 1, 0), K.CONV_BWD_DATA, 0, "stream_f32_k", 1),
    ((4, 4104, 128, 128, 256, 1, 1, 0), K.CONV_FWD, 0, "stream_f32_k", 0),
    ((32, 64, 112, 112, 48, 1, 1, 0), K.CONV_FWD, 0, "stream_f32_k", 0),
    # ... and where a slice of channels or a tile of results would not be full, in place or in tiles, with room too
    ((217, 16, 62, 62, 40, 1, 1, 0), K.CONV_FWD, 1.0, "stream_f32_k", 0),
    ((205, 56, 59, 59, 48, 1, 1, 0), K.CONV_FWD, 1.0, "stream_f32_k", 0),
    ((84, 64, 56, 56, 56, 1, 1, 0), K.CONV_FWD, 1.0, "conv_f32_gather_uniform", None),
    ((60, 40, 60, 60, 200, 1, 1, 0), K.CONV_FWD, 1.0, "conv_f32_gather_uniform", None),
    ((109, 64, 62, 62, 352, 1, 1, 0), K.CONV_FWD, 1.0, "stream_f32_k_window", None),
    # no room for three parts, but for the filter as it is; not for that either
    ((8, 512, 14, 14, 512, 3, 1, 1), K.CONV_FWD, 1.0, "stream_f32_k_window", None),
    ((8, 512, 14, 14, 512, 3, 1, 1), K.CONV_FWD, 4 * 9 * 512 * 512, "stream_f32_k", 3),
    ((8, 512, 14, 14, 512, 3, 1, 1), K.CONV_BWD_DATA, 4 * 9 * 512 * 512, "stream_f32_k", 3),
    ((8, 64, 28, 28, 64, 3, 1, 1), K.CONV_FWD, 64, "stream_f32_k", 2),
    ((256, 64, 56, 56, 64, 3, 1, 1), K.CONV_FWD, 1.0, "stream_f32_k_window", None),
    ((256, 64, 56, 56, 64, 3, 1, 1), K.CONV_FWD, 6 * 9 * 64 * 64 - 16, "conv_f32_gather_uniform", None),
    # windows that would leave the chip half empty
    ((103, 40, 13, 13, 64, 3, 2, 1), K.CONV_FWD, 1.0, "stream_f32_k", 3),
    ((1, 16, 107, 107, 336, 3, 1, 1), K.CONV_BWD_DATA, 1.0, "stream_f32_k", 3),
    ((29, 72, 37, 37, 16, 3, 1, 1), K.CONV_FWD, 1.0, "stream_f32_k", 3),
    ((3, 128, 54, 54, 72, 3, 1, 1), K.CONV_BWD_DATA, 1.0, "stream_f32_k", 3),
    ((141, 16, 48, 48, 296, 3, 2, 1), K.CONV_FWD, 1.0, "stream_f32_k", 3),
    # what windows do not take at all
    ((243, 8, 32, 32, 288, 5, 2, 2), K.CONV_FWD, 1.0, "stream_f32_k", 3),
    ((2, 456, 15, 15, 40, 7, 1, 3), K.CONV_FWD, 1.0, "stream_f32_k", 3),
]


@on_stub
def test_fp32_routes():
    for shape, kind, room, kernel, reads in F32_ROUTES:
        launches = convolution(kind, shape, K.FLOAT, room=room)[0]
        (ran,) = [x for x in launches if "pack" not in x[0] and "build" not in x[0]]
        assert ran[0] == kernel and reads in (None, ran[1][1]), (shape, kind, room, ran)


@on_stub
def test_fp32_windows_of_25_taps():
    """Blocks of four wavefronts along the pixels from 560 tiles on; fewer share the reduction."""
    for images, four in ((32, False), (45, False), (46, True), (64, True)):
        _, (name, _, blocks, _) = convolution(K.CONV_FWD, (images, 32, 14, 14, 64, 5, 1, 2), K.FLOAT)[0]
        assert name == "stream_f32_k_window" and (blocks == -(-images * 196 // 128) * 2) == four, (images, blocks)


@on_stub
def test_fp32_1x1_filters_that_a_program_packs():
    """Size of the copy: in three parts for windows, as it is where they cannot be, none where the filter in place is as good."""
    for shape, floats in (((24, 64, 56, 56, 64, 1, 1, 0), 6 / 4 * 64 * 64), ((32, 64, 56, 56, 64, 1, 1, 0), 0), ((12, 96, 40, 40, 24, 1, 1, 0), 0),
                          ((4, 96, 40, 40, 24, 1, 1, 0), 6 / 4 * 32 * 96), ((12, 24, 40, 40, 144, 1, 1, 0), 160 * 24), ((4, 2048, 7, 7, 512, 1, 1, 0), 6 / 4 * 512 * 2048),
                          ((96, 64, 56, 56, 64, 1, 1, 0), 0), ((8, 256, 56, 56, 512, 1, 2, 0), 6 / 4 * 512 * 256)):
        n, c, h, w, k, r, stride, pad = shape
        views = []
        for a, d in ((X, (n, c, h, w)), (W, (k, c, r, r)), (Y, (n, k, (h - 1) // stride + 1, (w - 1) // stride + 1))):
            v = image(a, *d, dtype=K.FLOAT)
            v.strides[:] = [d[1] * d[2] * d[3], d[2] * d[3], d[3], 1]
            views.append(C.byref(v))
        assert K.lib().saga_hip_conv2d_pack_bytes(K.CONV_FWD, *views, C.byref(K.ConvParams(pad, stride, 1, 1))) == 4 * floats, shape
