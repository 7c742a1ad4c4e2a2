// fp16 channels-last convolutions (forward and backward data) for grids too small to fill the chip with the LDS-tiled
// kernels of conv_mfma.hip.  See stream_f16.hip.
#pragma once
#include "common.hpp"

struct StreamF16 {
    const half_t *a; // gathered tensor, rows of lda halves
    const half_t *b; // filter rows [N][R][S][C]
    half_t *out;     // rows of ldo halves
    unsigned a_bytes, b_bytes;
    int batch, N, C; // images, output channels, channels of the gathered tensor (a multiple of 8)
    int IH, IW, OH, OW, R, S, pad, stride, dil, lda, ldo;
    int bwd;         // backward data: stride and dilation act on the output side
    float alpha, beta;
    const half_t *bias; // optional, alpha == 1: per output channel, added to the product
    // forward, optional: y = act(v * sc + sh (+ z)), sc = s*rsqrt(v+eps), sh = b - m*sc
    const float *bn_s, *bn_b, *bn_m, *bn_v;
    float bn_eps;
    int bn_flags;
    const half_t *z;
    int ldz;
    // optional: per row of blocks and channel two sums over the stored values v, [rows][N][2]: of v and v*v, or, where the
    // output is the gradient of a batch norm's (+ relu) result and bq_x that norm's input x, of v and v * (x - mean) with v
    // masked by the relu first (what conv_gather_gemm_dma's epilogues leave)
    float *sums;
    const half_t *bq_x;
    int bq_ldx, bq_relu;
    const float *bq_mean, *bq_s, *bq_invstd, *bq_b;
    unsigned out_bytes, z_bytes, bq_bytes; // (set by the launch)
};

// Blocks that share the reduction of each of `tiles` tiles of the tiled kernels (256 pixels x bn channels); conv_mfma.hip.
int conv_tile_split(int64_t tiles, int bn, int slices);
// Whether this kernel is the faster one for the problem.
bool stream_f16_wanted(const StreamF16 &g);
// Rows of sums a launch writes at most (by batch, N, C, OH, OW, R, S, stride and bwd); 0 if it is not wanted.
int stream_f16_sum_rows(const StreamF16 &g);
// SAGA_HIP_EUNSUPPORTED (nothing enqueued) outside what it covers.
int stream_f16_launch(const StreamF16 &g, hipStream_t st, int *sum_rows);
