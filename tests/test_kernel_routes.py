"""Which kernels the library's entry points launch, and what they refuse, without a GPU (over the stub runtime)."""
import ctypes as C

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
