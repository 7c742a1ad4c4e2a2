// Backward filter of fp32 3x3, stride-1 convolutions on the bf16 matrix unit (filter_f32.hip).
#pragma once
#include "conv.hpp"

struct FilterWindows {
    int pairs = 0;  // blocks of output channels times blocks of input channels; 0: not this kernel's
    int splits = 0; // partial results: shares of the tiles
    int kb, cb;     // output and input channels of a block
    int rows;       // of a tile, of 8 columns
    int tiles;      // of all images
};
FilterWindows plan_filter_windows(const ConvGeom &g);
double filter_windows_ns(const FilterWindows &p, const ConvGeom &g); // what it takes
// partial[splits][K][9][C]; splits may be fewer than planned.  SAGA_HIP_EUNSUPPORTED: nothing was launched.
int launch_filter_windows(const FilterWindows &p, const SagaTensorView *x, const SagaTensorView *dy, float *partial, const ConvGeom &g,
                          hipStream_t st);
