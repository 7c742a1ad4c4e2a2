// fp32 convolutions of one to four input channels, forward (thin_f32.hip)
#pragma once
#include "conv.hpp"

// SAGA_HIP_EUNSUPPORTED (nothing enqueued) outside what the kernel covers
int thin_f32_conv(const SagaTensorView *x, const SagaTensorView *w, const SagaTensorView *y, const ConvGeom &g, float alpha,
                  float beta, const StreamEpilogue &e, hipStream_t st, bool pool = false);
// with a max pooling of 2x2 windows behind it (pool), whose output y is
bool thin_f32_maxpool_ok(const SagaTensorView *x, const SagaTensorView *w, const SagaTensorView *y, const ConvGeom &g);
