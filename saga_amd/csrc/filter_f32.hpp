// Backward filter of fp32 3x3, stride-1 convolutions on the bf16 matrix unit (filter_f32.hip).
#pragma once
#include "conv.hpp"

struct FilterWindows {
    int pairs;  // blocks of 64 output channels times blocks of 64 input channels; 0: not this kernel's
    int splits; // partial results: shares of the tiles
};
FilterWindows plan_filter_windows(const ConvGeom &g);
double filter_windows_ns(const FilterWindows &p, const ConvGeom &g); // what it takes
// partial[splits][K][9][C]; splits may be fewer than planned.  SAGA_HIP_EUNSUPPORTED: nothing was launched.
int launch_filter_windows(const FilterWindows &p, const SagaTensorView *x, const SagaTensorView *dy, float *partial, const ConvGeom &g,
                          hipStream_t st);
