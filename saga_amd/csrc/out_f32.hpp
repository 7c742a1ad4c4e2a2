// How the fp32 kernels with 32x32 matrix instructions leave their results: fours of channels of one pixel per lane.
#pragma once
#include "stream_f32.hpp"

constexpr unsigned OUT_NOWHERE = 0x7fffff00u; // behind every buffer: loads return zero, stores do nothing

// division by a constant of the launch, of numbers below 2^31
struct FastDiv {
    unsigned d, mul, shift;
    __device__ __forceinline__ int div(int n) const { return d == 1 ? n : (int)(__umulhi((unsigned)n, mul) >> shift); }
};

inline FastDiv fast_div(int d)
{
    FastDiv f = {(unsigned)d, 0, 0};
    if(d > 1) {
        const int l = 32 - __builtin_clz(d - 1);
        f.mul = (unsigned)((1ull << (31 + l)) / d + 1);
        f.shift = l - 1;
    }
    return f;
}

// bytes from a tensor's first element to the end of its last; -1: a negative stride
inline long long extent_of(const SagaTensorView *v)
{
    long long n = 1;
    for(int i = 0; i < 4; i++) {
        if(v->strides[i] < 0)
            return -1;
        n += (v->dims[i] - 1) * v->strides[i];
    }
    return n * 4;
}

struct OutArgs {
    float *out;
    unsigned o_bytes, z_bytes;
    int N; // channels
    long long o_sn, o_sc, o_sh, o_sw;
    float alpha, beta;
    EpilogueF32 e;
};

// false: out of the reach of 32-bit offsets
inline bool describe_out(const SagaTensorView *out, float alpha, float beta, const StreamEpilogue &e, OutArgs &a)
{
    const long long o = extent_of(out), z = e.z ? extent_of(e.z) : 0;
    if(o < 0 || z < 0 || o > OUT_NOWHERE || z > OUT_NOWHERE)
        return false;
    a.out = (float *)out->ptr;
    a.o_bytes = (unsigned)o;
    a.z_bytes = (unsigned)z;
    a.N = out->dims[1];
    a.o_sn = out->strides[0]; a.o_sc = out->strides[1]; a.o_sh = out->strides[2]; a.o_sw = out->strides[3];
    a.alpha = alpha;
    a.beta = beta;
    a.e = epilogue_f32(e);
    return true;
}

struct Four {
    float v[4];
};

// Pixel m of a convolution's output: rows one after the other, or, POOL, the 2x2 windows of a max pooling (ow and oh count those), four
// neighbouring lanes each in the order in which they are compared.
template <bool POOL> __device__ __forceinline__ void place_pixel(const FastDiv &ow, const FastDiv &oh, int m, int &n, int &oy, int &ox)
{
    const int at = POOL ? m >> 2 : m, t = ow.div(at);
    ox = at - t * (int)ow.d;
    n = oh.div(t);
    oy = t - n * (int)oh.d;
    if(POOL) {
        ox = 2 * ox + (m & 1);
        oy = 2 * oy + ((m >> 1) & 1);
    }
}

// Everything per lane is in the vector offset, everything per value in the scalar one; a pixel or a channel that is not
// there gets an offset behind the buffer.  EX: there is something to add to the values or to apply to them.  POOL: the largest of a window's
// four goes out, in the place of its four pixels; the lanes of a window exchange them and store one channel each.
template <bool EX, bool POOL = false> struct FourOut {
    const OutArgs &g;
    __amdgpu_buffer_rsrc_t ro, rz;
    unsigned osc4, zsc4;
    int fk; // the lane's half: channels 4 * fk on of every eight

    __device__ __forceinline__ FourOut(const OutArgs &a, int fk_) : g(a), fk(fk_)
    {
        ro = __builtin_amdgcn_make_buffer_rsrc((void *)g.out, 0, (int)g.o_bytes, 0x00020000);
        rz = __builtin_amdgcn_make_buffer_rsrc((void *)(EX ? g.e.z : nullptr), 0, EX ? (int)g.z_bytes : 0, 0x00020000);
        osc4 = (unsigned)(g.o_sc * 4);
        zsc4 = EX ? (unsigned)(g.e.z_sc * 4) : 0;
    }
    __device__ __forceinline__ unsigned out_at(bool ok, int n, int y, int x) const
    {
        if constexpr(POOL)
            return ok ? (unsigned)((n * g.o_sn + (y >> 1) * g.o_sh + (x >> 1) * g.o_sw + (4 * fk + (threadIdx.x & 3)) * g.o_sc) * 4) : OUT_NOWHERE;
        return ok ? (unsigned)((n * g.o_sn + y * g.o_sh + x * g.o_sw + 4 * fk * g.o_sc) * 4) : OUT_NOWHERE;
    }
    // of the window of four lanes, which run along it (the rule of the pooling kernels: what is not at most the largest so far, and a
    // NaN stays)
    __device__ __forceinline__ static float largest(float x)
    {
        const int i = __builtin_bit_cast(int, x);
        float most = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, i, 0x00, 0xf, 0xf, true));
        const float others[3] = {__builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, i, 0x55, 0xf, 0xf, true)),
                                 __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, i, 0xaa, 0xf, 0xf, true)),
                                 __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, i, 0xff, 0xf, 0xf, true))};
#pragma unroll
        for(int k = 0; k < 3; k++)
            most = !(others[k] <= most) && most == most ? others[k] : most;
        return most;
    }
    __device__ __forceinline__ unsigned z_at(bool ok, int n, int y, int x) const
    {
        return EX && ok ? (unsigned)((n * g.e.z_sn + y * g.e.z_sh + x * g.e.z_sw + 4 * fk * g.e.z_sc) * 4) : OUT_NOWHERE;
    }
    // channels n + 4 * fk ... of a tensor (the scalar offset stays inside; channels behind the last are not stored)
    __device__ __forceinline__ Four fetch(__amdgpu_buffer_rsrc_t r, unsigned pos, unsigned step, int n) const
    {
        Four f;
#pragma unroll
        for(int j = 0; j < 4; j++)
            f.v[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, n + 4 * fk + j < g.N ? pos : OUT_NOWHERE,
                                                                                  n + j < g.N ? (n + j) * step : 0, 0));
        return f;
    }
    __device__ __forceinline__ Four before(unsigned pos, int n) const { return EX && g.beta != 0.0f ? fetch(ro, pos, osc4, n) : Four{}; }
    __device__ __forceinline__ Four residual(unsigned pos, int n) const { return EX && g.e.z ? fetch(rz, pos, zsc4, n) : Four{}; }
    // chan: scale and shift of channel n + 4 * fk on (read for an affine epilogue)
    __device__ __forceinline__ void store(unsigned pos, int n, const Four &val, const Four &was, const Four &res, const float *chan_scale,
                                          const float *chan_shift) const
    {
        float4_t scale = {1, 1, 1, 1}, shift = {0, 0, 0, 0};
        if(EX && g.e.affine()) {
            scale = *(const float4_t *)chan_scale;
            shift = *(const float4_t *)chan_shift;
        }
        if constexpr(POOL) {
            const int e = threadIdx.x & 3;
            float own = 0.0f;
#pragma unroll
            for(int j = 0; j < 4; j++) {
                const float most = largest(g.e.apply(val.v[j] * g.alpha, scale[j], shift[j], 0.0f));
                own = e == j ? most : own;
            }
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, own), ro, n + 4 * fk + e < g.N ? pos : OUT_NOWHERE,
                                                  n < g.N ? n * osc4 : 0, 0);
            return;
        }
#pragma unroll
        for(int j = 0; j < 4; j++) {
            float x = val.v[j] * g.alpha;
            if constexpr(EX) {
                if(g.beta != 0.0f)
                    x += g.beta * was.v[j];
                x = g.e.apply(x, scale[j], shift[j], res.v[j]);
            }
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, x), ro, n + 4 * fk + j < g.N ? pos : OUT_NOWHERE,
                                                  n + j < g.N ? (n + j) * osc4 : 0, 0);
        }
    }
};
