"""fp16 convolutions on small grids in steps of 64 channels: every tile that takes them, at sizes that end inside its pixels, its channels
and the wavefronts' shares of the reduction, on the whole numbers of test_gpu_ragged_channels: results are exact."""
import ctypes as C

import pytest
import torch

from saga_amd import kernels as K
from tests import stub_gpu, test_gpu_ragged_channels as rows
from tests.stub_gpu import on_stub

# as there; and the forward launch: tile, 32 channels to a step, steps of the ring (0: operands), wavefronts
SHAPES = {
    (1, 64, 5, 5, 33, 3, 1, 0, 0): (1, 1, 2, 4, 4),        # nine steps over four wavefronts
    (1, 512, 7, 7, 19, 3, 1, 1, 1): (1, 1, 2, 4, 4),
    (3, 192, 14, 13, 77, 3, 2, 0, 1): (1, 1, 2, 4, 4),     # three steps to a tap; backward: residue classes
    (4, 256, 14, 14, 251, 3, 1, 0, 0): (2, 2, 2, 2, 4),
    (1, 512, 21, 21, 1027, 3, 1, 0, 1): (4, 2, 2, 0, 8),
    (1, 256, 42, 42, 517, 3, 1, 2, 0): (4, 4, 2, 2, 4),
    (9, 64, 27, 26, 255, 5, 1, 3, 1): (4, 4, 2, 2, 4),     # two wavefronts along the pixels
    (5, 96, 14, 14, 130, 3, 1, 0, 0): (2, 2, 1, 4, 4),     # 64 channels do not divide these
}


@on_stub
def test_the_forms_they_are_for():
    L = K.lib()
    for shape, form in SHAPES.items():
        n, c, h, w, k, r, stride, wide, shift = shape
        ch = lambda *d: torch.empty(*d, dtype=torch.float16, device="meta").contiguous(memory_format=torch.channels_last)
        tensors = ch(n, c, h, w), ch(k, c, r, r), ch(n, k + wide, *rows.out_size(shape))[:, :k]
        views = [K.TensorView() for _ in range(3)]
        for v, t, at in zip(views, tensors, (1 << 20, 1 << 31, (1 << 30) + 2 * shift)):
            v.ptr, v.dtype = at, K.HALF
            v.dims[:], v.strides[:] = list(t.shape), list(t.stride())
        a, p = [C.byref(v) for v in views], C.byref(K.ConvParams(r // 2, stride, 1, 1))
        room = L.saga_hip_conv2d_workspace_size(K.CONV_FWD, *a, p)
        stub_gpu.launched()
        assert L.saga_hip_conv2d_fwd(*a, p, 1.0, 0.0, 1 << 32, room, None) == 0
        kernel, args, _, threads = stub_gpu.launched()[-1]
        assert (kernel, args[:4], threads) == ("stream_f16_k", form[:4], 64 * form[4]), (shape, kernel, args, threads)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_forward(shape):
    rows.test_forward(shape)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_backward(shape):
    rows.test_backward(shape)
