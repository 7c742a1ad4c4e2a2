// fp32 matrix products on v_mfma_f32_32x32x2_f32 straight from global memory: convolutions (forward and backward data)
// and the fully connected layers' GEMMs.  See stream_f32.hip.
#pragma once
#include "conv.hpp"

// StreamEpilogue as the kernels take it.  A block fetches the raw parameters of its channels before its main loop (fetch), one
// channel per thread, and leaves scale and shift in LDS after it (leave): four dependent loads per output value would
// cost more than the convolution's last step.  A norm of its own reads and writes the tensor once more in a launch of
// 7 - 25 us: 53 of them folded took a fp32 ResNet-50 batch of 8 from 2.12 to 1.79 ms.
struct EpilogueF32 {
    const float *bias, *bn_s, *bn_b, *bn_m, *bn_v, *z;
    float bn_eps;
    int relu;
    long long z_sn, z_sc, z_sh, z_sw;
    struct Raw {
        float s = 1, b = 0, m = 0, v = 0;
    };
    __device__ __forceinline__ bool affine() const { return bias || bn_s; }
    __device__ __forceinline__ Raw fetch(int n) const
    {
        Raw r;
        if(bn_s)
            r.s = bn_s[n], r.b = bn_b[n], r.m = bn_m[n], r.v = bn_v[n];
        else if(bias)
            r.b = bias[n];
        return r;
    }
    __device__ __forceinline__ void leave(const Raw &r, float &scale, float &shift) const
    {
        scale = bn_s ? r.s * rsqrtf(r.v + bn_eps) : 1.0f;
        shift = r.b - r.m * scale;
    }
    __device__ __forceinline__ float apply(float v, float scale, float shift, float residual) const
    {
        if(affine())
            v = __builtin_fmaf(v, scale, shift);
        if(z)
            v += residual;
        return relu && v == v ? fmaxf(v, 0.0f) : v;
    }
};

inline EpilogueF32 epilogue_f32(const StreamEpilogue &e)
{
    EpilogueF32 d = {e.bias, e.bn_s, e.bn_b, e.bn_m, e.bn_v, nullptr, e.bn_eps, e.relu, 0, 0, 0, 0};
    if(e.z) {
        d.z = (const float *)e.z->ptr;
        d.z_sn = e.z->strides[0]; d.z_sc = e.z->strides[1]; d.z_sh = e.z->strides[2]; d.z_sw = e.z->strides[3];
    }
    return d;
}

// bytes of workspace for a convolution; 0 when it needs none
size_t stream_f32_conv_workspace(bool bwd, const SagaTensorView *a, const SagaTensorView *out, const ConvGeom &g);
// a: x or dy, out: y or dx; packed (may be null): what stream_f32_pack left, otherwise packed into ws where needed.  SAGA_HIP_EUNSUPPORTED (nothing enqueued) outside what the kernel covers.
int stream_f32_conv(bool bwd, const SagaTensorView *a, const SagaTensorView *w, const SagaTensorView *out, const ConvGeom &g,
                    float alpha, float beta, const StreamEpilogue &e, const void *packed, void *ws, size_t ws_bytes, hipStream_t st,
                    bool pool = false); // pool: and a max pooling of 2x2 windows, whose output `out` is, where windows (below) do that
// whether a convolution is done in windows (window_f32.hip), of a filter packed beforehand or with that much workspace to pack it
bool stream_f32_windows(bool bwd, const SagaTensorView *a, const SagaTensorView *out, const ConvGeom &g, bool packed, size_t room,
                        bool pool = false);
// the filter in the order that the kernel loads it: bytes (0: not for this convolution), jobs (at most 16), launch
size_t stream_f32_packed_bytes(bool bwd, const SagaTensorView *a, const SagaTensorView *w, const SagaTensorView *out, const ConvGeom &g);
int stream_f32_pack_jobs(bool bwd, const SagaTensorView *w, const ConvGeom &g, void *packed, SagaFilterPackJob *jobs);
int stream_pack_blocks(const SagaFilterPackJob &j); // of stream_f32_pack
int stream_f32_pack(const SagaFilterPackJob *jobs, int njobs, int blocks, hipStream_t st);
// row-major C[M][N] = alpha * op(A) * op(B) + beta * C, bias per column of C
int stream_f32_gemm(int tA, int tB, int M, int N, int K, float alpha, const float *A, int lda, const float *B, int ldb,
                    float beta, float *C, int ldc, const float *bias, int relu, hipStream_t st);
