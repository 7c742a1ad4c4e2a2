// fp32 convolutions whose input positions are split and staged once per slice of channels (window_f32.hip)
#pragma once
#include "stream_f32.hpp"

// a convolution with one class of pixels: taps, position of pixel (0, 0) under the first, positions per pixel and per tap
struct WindowConv {
    int Tr, Ts, iy0, ix0, istep, tstep;
    unsigned a_bytes; // of the tensor read
};

// whether any such convolution of so many channels, input and output pixels could, whatever the number and the strides of its images
bool window_f32_may(const WindowConv &c, int channels, int IH, int IW, int OH, int OW);
// whether such a convolution goes through the kernel (with operands of the usual extent)
// (pool: out is what a max pooling of 2x2 windows makes of the convolution's)
bool window_f32_takes(const WindowConv &c, const SagaTensorView *a, const SagaTensorView *out, bool pool);
// packed: the filter as stream_f32_pack leaves it.  SAGA_HIP_EUNSUPPORTED (nothing enqueued) outside what the kernel covers.
int window_f32_conv(const WindowConv &c, const SagaTensorView *a, const SagaTensorView *out, float alpha, float beta,
                    const StreamEpilogue &e, const void *packed, size_t packed_bytes, bool pool, hipStream_t st);
