"""Max pooling over 2x2 and 3x3 windows (csrc/pool.hip, pool_max_k): which kernel runs on either side of 2^30 results, on the stub
runtime; on the GPU windows that lie in part or wholly in the padding."""
import ctypes as C

import pytest
import torch

from saga_amd import kernels as K
from tests import stub_gpu
from tests.stub_gpu import on_stub


@pytest.mark.parametrize("images,kernel", [(63, "pool_max_k"), (64, "pool_fwd_k")])
@on_stub
def test_32_bit_work_indices(images, kernel):
    def view(address, h, w):
        v = K.TensorView()
        v.ptr, v.dtype = address, K.FLOAT
        v.dims[:], v.strides[:] = [images, 64, h, w], [64 * h * w, h * w, w, 1]
        return v

    x, y = view(1 << 20, 513, 513), view(1 << 40, 512, 512)
    stub_gpu.launched()
    assert K.lib().saga_hip_pool_fwd(K.POOL_MAX, C.byref(x), C.byref(y), None, 2, 0, 1, None) == 0
    assert [name for name, *_ in stub_gpu.launched()] == [kernel]


def reference(x, size, pad, stride):
    """Maxima in row-major order of positions, the first of equal ones and of NaNs; without a position -inf and -1."""
    n, c, h, w = x.shape
    p, q = 1 + (h + 2 * pad - size) // stride, 1 + (w + 2 * pad - size) // stride
    y, at = torch.full((n, c, p, q), float("-inf")), torch.full((n, c, p, q), -1, dtype=torch.int32)
    for i in range(p):
        for j in range(q):
            for r in range(i * stride - pad, i * stride - pad + size):
                for s in range(j * stride - pad, j * stride - pad + size):
                    if 0 <= r < h and 0 <= s < w:
                        v, best = x[:, :, r, s], y[:, :, i, j]
                        take = (at[:, :, i, j] < 0) | (~(v <= best) & ~best.isnan())
                        y[:, :, i, j] = torch.where(take, v, best)
                        at[:, :, i, j] = torch.where(take, r * w + s, at[:, :, i, j])
    return y, at


@pytest.mark.gpu
@pytest.mark.parametrize("size,pad,stride,h,w", [(2, 0, 2, 8, 6), (2, 1, 1, 3, 5), (2, 3, 2, 4, 3), (3, 1, 2, 7, 9), (3, 4, 1, 2, 1), (3, 5, 3, 5, 4)])
@pytest.mark.parametrize("layout", ["nchw", "nhwc"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16], ids=str)
def test_windows_in_the_padding(dtype, layout, size, pad, stride, h, w):
    g = torch.Generator().manual_seed(size + pad)
    x = torch.randint(-9, 10, (3, 16, h, w), generator=g).float()
    x[0, 1, h // 2, w // 2], x[1, 2, 0, 0], x[2, 3] = float("nan"), float("inf"), float("-inf")
    want, at = reference(x, size, pad, stride)
    fmt = torch.channels_last if layout == "nhwc" else torch.contiguous_format
    xd = x.to("cuda", dtype).contiguous(memory_format=fmt)
    yd = torch.full(want.shape, 7.0, device="cuda", dtype=dtype).contiguous(memory_format=fmt)
    idx = torch.full(want.shape, 7, device="cuda", dtype=torch.int32).contiguous(memory_format=fmt)
    K.check(K.lib().saga_hip_pool_fwd(K.POOL_MAX, *(C.byref(K.view(t)) for t in (xd, yd, idx)), size, pad, stride, K.stream_ptr()))
    assert torch.equal(yd.float().cpu().nan_to_num(77.0), want.nan_to_num(77.0)) and torch.equal(yd.isnan().cpu(), want.isnan())
    assert torch.equal(idx.cpu(), at)
