// fp32 matrix products on v_mfma_f32_32x32x2_f32 straight from global memory: convolutions (forward and backward data)
// and the fully connected layers' GEMMs.  See stream_f32.hip.
#pragma once
#include "conv.hpp"

// Per output channel (or GEMM row) and element, after alpha and beta: out = act(v * scale + shift + z).
struct StreamEpilogue {
    const float *bias = nullptr;                                                    // shift
    const float *bn_s = nullptr, *bn_b = nullptr, *bn_m = nullptr, *bn_v = nullptr; // scale = s*rsqrt(v+eps), shift = b - m*scale
    float bn_eps = 0;
    const SagaTensorView *z = nullptr;
    int relu = 0;
};

// bytes of workspace for a convolution; 0 when it needs none
size_t stream_f32_conv_workspace(bool bwd, const ConvGeom &g);
// a: x or dy, out: y or dx.  SAGA_HIP_EUNSUPPORTED (nothing enqueued) outside what the kernel covers.
int stream_f32_conv(bool bwd, const SagaTensorView *a, const SagaTensorView *w, const SagaTensorView *out, const ConvGeom &g,
                    float alpha, float beta, const StreamEpilogue &e, void *ws, size_t ws_bytes, hipStream_t st);
// row-major C[M][N] = alpha * op(A) * op(B) + beta * C, bias per column of C
int stream_f32_gemm(int tA, int tB, int M, int N, int K, float alpha, const float *A, int lda, const float *B, int ldb,
                    float beta, float *C, int ldc, const float *bias, int relu, hipStream_t st);
