// Backward filter of 3x3, stride-1 convolutions, image strips in LDS (filter_strips.hip).
#pragma once
#include "conv.hpp"

struct FilterStrips {
    int tw, nst;    // columns of a tile, row pairs of a group of wavefronts; nst 0: not this kernel's
    int pairs;      // blocks of 64 output channels times blocks of 64 input channels
    int splits;     // partial results: shares of the tiles
};
// g.C, g.K: as the kernel sees them (multiples of 8); other_ns: what the other kernel takes
FilterStrips plan_filter_strips(const ConvGeom &g, int cus, double other_ns);
static inline size_t filter_strips_bytes(const FilterStrips &p, const ConvGeom &g)
{
    return p.nst ? (size_t)p.splits * g.K * 9 * g.C * sizeof(float) : 0;
}
// partial[splits][K][9][C]; x, dy: pixel pitches ldx, ldy, 16-byte aligned
int launch_filter_strips(const FilterStrips &p, const half_t *x, int64_t ldx, const half_t *dy, int64_t ldy, float *partial,
                         const ConvGeom &g, hipStream_t st);
