// Internal interfaces between the convolution dispatcher and its kernel families.
#pragma once
#include "common.hpp"

struct ConvGeom {
    int N, C, H, W;    // input (x / dx)
    int K, R, S;       // filters
    int P, Q;          // output (y / dy)
    int pad, stride, dil, group;
};

// Direct (non-MFMA) kernels: any dtype in {half, float}, any strides, groups, dilation.
int conv_direct_fwd(const SagaTensorView *x, const SagaTensorView *w, const SagaTensorView *y, const ConvGeom &g,
                    float alpha, float beta, hipStream_t st);
int conv_direct_bwd_data(const SagaTensorView *dy, const SagaTensorView *w, const SagaTensorView *dx,
                         const ConvGeom &g, float alpha, float beta, hipStream_t st);
int conv_direct_bwd_filter(const SagaTensorView *x, const SagaTensorView *dy, const SagaTensorView *dw,
                           const ConvGeom &g, float alpha, float beta, hipStream_t st);

// MFMA implicit-GEMM kernels (fp16, channels-last).  Each returns SAGA_HIP_EUNSUPPORTED when the
// problem is outside what it covers, and the dispatcher falls back to the direct kernels.
size_t conv_mfma_workspace(int kind, const SagaTensorView *x, const SagaTensorView *w, const SagaTensorView *y,
                           const ConvGeom &g);
// stats (optional): receives per block row and output channel the sum and the sum of squares of
// the stored outputs, [*stats_rows][K][2] floats; needs beta == 0 and conv_mfma_stats_floats(g) floats
size_t conv_mfma_stats_floats(const ConvGeom &g);
// bias (optional, fp16, alpha == 1): *bias_done says whether the launch added it
// batch-norm inference (+ residual + relu) folded into the forward epilogue
struct ConvBnFold {
    const float *s, *b, *m, *v;
    float eps;
    int flags;
    const SagaTensorView *z;
};
int conv_mfma_fwd(const SagaTensorView *x, const SagaTensorView *w, const SagaTensorView *y, const ConvGeom &g,
                  float alpha, float beta, void *ws, size_t ws_bytes, hipStream_t st, float *stats = nullptr,
                  size_t stats_floats = 0, int *stats_rows = nullptr, const ConvBnFold *bn = nullptr, const void *bias = nullptr,
                  bool *bias_done = nullptr, const void *packed = nullptr);
// The same with a norm, relu and max pooling behind it, in one launch (stem_f16.hip); y: the pooled tensor.  ok: whether there is one
// for tensors like these.
bool conv_bn_maxpool_ok(const SagaTensorView *x, const SagaTensorView *w, const SagaTensorView *y, const ConvGeom &g, int size,
                        int pool_pad, int pool_stride);
int conv_bn_maxpool(const SagaTensorView *x, const SagaTensorView *w, const SagaTensorView *y, const ConvGeom &g, const float *s,
                    const float *b, const float *m, const float *v, float eps, int size, int pool_pad, int pool_stride, hipStream_t st);
// bytes of the packed filter that a forward launch on these tensors reads (window_f16.hip); 0: none
size_t conv_mfma_packed_bytes(const SagaTensorView *x, const SagaTensorView *w, const SagaTensorView *y, const ConvGeom &g);
void conv_mfma_pack_job(const SagaTensorView *w, const ConvGeom &g, void *packed, SagaFilterPackJob &job);
// backward data whose result dx is the gradient of a batch norm's (+ relu) output, with that norm's first
// backward pass done in the epilogue: dx is stored masked by the relu and partial[*partial_rows][C][2]
// receives sum(dx) and sum(dx * (x - mean)) per block row and channel.  EUNSUPPORTED (nothing written)
// outside the pipelined kernel with 16-byte channel vectors.
struct ConvBnBwdLink {
    const SagaTensorView *x;               // the norm's input, dims of dx
    const float *mean, *invstd, *s, *b;    // invstd, s, b only for relu
    int relu;
    float *partial;
    size_t partial_floats;                 // at least conv_mfma_bnbwd_floats(g)
    int *partial_rows;
};
size_t conv_mfma_bnbwd_floats(const ConvGeom &g);
int conv_mfma_bwd_data(const SagaTensorView *dy, const SagaTensorView *w, const SagaTensorView *dx,
                       const ConvGeom &g, float alpha, float beta, void *ws, size_t ws_bytes, hipStream_t st,
                       const void *wt_ready = nullptr, const ConvBnBwdLink *link = nullptr, const void *bias = nullptr,
                       bool *bias_done = nullptr);
bool conv_mfma_bwd_data_ok(const SagaTensorView *dy, const SagaTensorView *w, const SagaTensorView *dx, const ConvGeom &g);
bool conv_mfma_bnbwd_link_ok(const SagaTensorView *dy, const SagaTensorView *w, const SagaTensorView *dx, const ConvGeom &g);
int conv_mfma_transpose_blocks(int K, int C, int RS);
int conv_mfma_transpose_batched(const SagaFilterTransposeJob *jobs, int njobs, int total_blocks, hipStream_t st);
int conv_mfma_bwd_filter(const SagaTensorView *x, const SagaTensorView *dy, const SagaTensorView *dw,
                         const ConvGeom &g, float alpha, float beta, void *ws, size_t ws_bytes, hipStream_t st);

// fp32 MFMA implicit-GEMM kernels (any strides, groups == 1); SAGA_HIP_EUNSUPPORTED otherwise.
size_t conv_f32_workspace(int kind, const SagaTensorView *x, const SagaTensorView *w, const SagaTensorView *y,
                          const ConvGeom &g);
// Per output channel and element, after alpha and beta: out = act(v * scale + shift + z).
struct StreamEpilogue {
    const float *bias = nullptr;                                                    // shift
    const float *bn_s = nullptr, *bn_b = nullptr, *bn_m = nullptr, *bn_v = nullptr; // scale = s*rsqrt(v+eps), shift = b - m*scale
    float bn_eps = 0;
    const SagaTensorView *z = nullptr;
    int relu = 0;
};
int conv_f32_fwd(const SagaTensorView *x, const SagaTensorView *w, const SagaTensorView *y, const ConvGeom &g, float alpha,
                 float beta, void *ws, size_t ws_bytes, hipStream_t st, const StreamEpilogue &e = StreamEpilogue(),
                 const void *packed = nullptr);
// and a max pooling of 2x2 windows, whose output y is, in the same launch; packed: there is a packed filter
bool conv_f32_maxpool_ok(const SagaTensorView *x, const SagaTensorView *w, const SagaTensorView *y, const ConvGeom &g, bool packed);
int conv_f32_maxpool(const SagaTensorView *x, const SagaTensorView *w, const SagaTensorView *y, const ConvGeom &g, void *ws, size_t ws_bytes,
                     const StreamEpilogue &e, const void *packed, hipStream_t st);
int conv_f32_bwd_data(const SagaTensorView *dy, const SagaTensorView *w, const SagaTensorView *dx, const ConvGeom &g,
                      float alpha, float beta, void *ws, size_t ws_bytes, hipStream_t st, const StreamEpilogue &e = StreamEpilogue(),
                      const void *packed = nullptr);
// bytes of the packed filter that a launch on these tensors reads (see stream_f32.hip); 0: none
size_t conv_f32_packed_bytes(int kind, const SagaTensorView *x, const SagaTensorView *w, const SagaTensorView *y, const ConvGeom &g);
int conv_f32_bwd_filter(const SagaTensorView *x, const SagaTensorView *dy, const SagaTensorView *dw, const ConvGeom &g,
                        float alpha, float beta, void *ws, size_t ws_bytes, hipStream_t st);
