// The stem of an image network in inference: a 7x7 convolution at stride 2 over three channels, the folded batch norm, relu and
// the 3x3 max pooling at stride 2 behind it in one launch, fp16 channels-last.
//
// Between them lies the largest tensor of such a network (411 MB of a batch of 256 at 224x224), written and read for the sake of a
// quarter of its values; and the convolution by itself takes a copy of the image with four channels to a pixel and one of the
// filter in that order.  Here a block stages the rows of a strip of pooled rows as pixels of four channels (8 bytes, the last one
// zero) in LDS, straight from the image, and builds its operands of the filter, which stay in registers, once.
//
// A wavefront has 32 channels and up to 32 pooled columns.  Of two accumulators one is the convolution's even columns 2q, the
// other its odd ones 2q + 1, a lane each; a pooled row takes the convolution's rows 2p - 1 (kept from the row before), 2p and
// 2p + 1, which are reduced together, so that an operand from LDS serves both.  Rows and columns meet as packed halves: the
// largest of three rows, then of (even, odd, odd of the lane below).  The lane below lane 0 belongs to the group of columns
// before, whose last odd column lane 0 computes again instead; the first group, at the edge of the image, has 32 outputs, the
// others 31.  Positions outside the image count as zero: behind the relu nothing is less.
//
// A pixel's window is four 16-byte pieces, two pixels each, of a row; pieces of even and of odd number lie apart, so that the lanes of
// either half of a wavefront, two pieces apart, read consecutive addresses.  A reduction of 32 per filter row (21 of them
// taps), row by row, as the kernel for the convolution alone (conv_thin_rows) has it: the same sums, rounded to fp16 as they
// were in between.
//
// us, the copies of image and filter, convolution and pooling that this replaces / this, 64 channels: 256x224x224 345 (of it the
// convolution 175) / 118, 12x200x200 about 55 / 15, 1x224x224 24 / 9.9.  Of the 118 the matrix instructions take 53 at 2.1 GHz; the
// rest is what the two blocks of a CU do not hide of each other: staging, norm and relu of four values for each that is
// stored, and the eighth of a wavefront's columns that an image of 224 leaves empty.
#include "conv.hpp"

#include <algorithm>

namespace {

constexpr int R = 7;

struct StemArgs {
    const half_t *x, *w;
    half_t *y;
    const float *s, *b, *m, *v;
    float eps;
    int H, W, P, Q, Pp, Qp, K, S, pad; // image; convolution's output; pooled output; channels; columns of the filter
    int x_bytes;                       // of an image
    int64_t ldy;
    int TP, strips, ntiles;            // pooled rows of a strip, strips of an image, of all
    int plane, row;                    // LDS bytes of every second piece of a row, and of a row
    int pieces;                        // of a row
    int items, groups, runs;           // what a block's wavefronts share: channels' halves x groups of columns x runs of rows
    int w_bytes, w_at;                 // the filter, and where it is staged
};

typedef unsigned uint2_t __attribute__((ext_vector_type(2)));
typedef unsigned uint4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) const uint4_t *lds_vec_t;

__device__ __forceinline__ half2_t halves(unsigned v) { return __builtin_bit_cast(half2_t, v); }
__device__ __forceinline__ unsigned largest(unsigned a, unsigned b, unsigned c) // (NaN where one of them is)
{
    return __builtin_bit_cast(unsigned, __builtin_elementwise_maximum(__builtin_elementwise_maximum(halves(a), halves(b)), halves(c)));
}

__global__ void __launch_bounds__(256, 2) conv7x7s2_bn_maxpool(StemArgs t)
{
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63, l = lane & 31, hi = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    {
        const uint4_t *src = (const uint4_t *)t.w;
        for(int i = tid; i < t.w_bytes / 16; i += 256)
            *(uint4_t *)(smem + t.w_at + i * 16) = src[i];
    }

    // Rows of a strip, as they lie in LDS.  A piece is two pixels, twelve bytes of an image row at an address that is a multiple of
    // two: two loads of eight bytes, each dword of which holds some of them, so that none reaches beyond the image's last.
    auto stage = [&](int tile) {
        const int n = tile / t.strips, p0 = (tile - n * t.strips) * t.TP;
        const int count = 4 * std::min(t.TP, t.Pp - p0) + R, h0 = 4 * p0 - 2 - t.pad; // image row of the first
        const uintptr_t first = (uintptr_t)(t.x + (int64_t)n * t.H * t.W * 3);
        const int shift = (int)(first & 2);
        const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void *)(first - shift), 0, (t.x_bytes + shift + 3) & ~3, 0x00020000);
        const int total = count * t.pieces, dr = 256 / t.pieces, dg = 256 - dr * t.pieces;
        int r = tid / t.pieces, g = tid - r * t.pieces;
        constexpr int U = 4;
        for(int i = tid; i < total; i += 256 * U) {
            uint2_t a[U], c[U];
            int to[U], odd[U];
            bool in0[U], in1[U];
#pragma unroll
            for(int u = 0; u < U; u++) {
                const int h = h0 + r, px = 2 * g - t.pad;
                const bool row = i + 256 * u < total && (unsigned)h < (unsigned)t.H;
                in0[u] = row && (unsigned)px < (unsigned)t.W;
                in1[u] = row && (unsigned)(px + 1) < (unsigned)t.W;
                to[u] = i + 256 * u < total ? r * t.row + (g & 1) * t.plane + (g >> 1) * 16 : -1;
                const int at = (h * t.W + px) * 6 + shift;
                odd[u] = at & 2;
                const unsigned off = (unsigned)(at & ~3);
                a[u] = __builtin_bit_cast(uint2_t, __builtin_amdgcn_raw_buffer_load_b64(rx, in0[u] ? off : 0x7fffff00u, 0, 0));
                c[u] = __builtin_bit_cast(uint2_t, __builtin_amdgcn_raw_buffer_load_b64(rx, in1[u] ? off + (odd[u] ? 8 : 4) : 0x7fffff00u, 0, 0));
                r += dr;
                g += dg;
                if(g >= t.pieces) {
                    g -= t.pieces;
                    r++;
                }
            }
#pragma unroll
            for(int u = 0; u < U; u++) {
                if(to[u] < 0)
                    continue;
                uint4_t v; // of the first pixel: a's bytes from `odd` on; of the second: odd, from c's dword 0 and 1, of a's last half
                const unsigned a0 = a[u][0], a1 = a[u][1], c0 = c[u][0], c1 = c[u][1];
                v[0] = odd[u] ? __builtin_amdgcn_alignbit(a1, a0, 16) : a0;
                v[1] = odd[u] ? a1 >> 16 : a1 & 0xffffu;
                v[2] = odd[u] ? c0 : __builtin_amdgcn_alignbit(c1, c0, 16);
                v[3] = odd[u] ? c1 & 0xffffu : c1 >> 16;
                if(!in0[u])
                    v[0] = v[1] = 0;
                if(!in1[u])
                    v[2] = v[3] = 0;
                *(uint4_t *)(smem + to[u]) = v;
            }
        }
    };
    const bool apart = t.w_at > 0; // (the filter has room of its own: both are on their way at once)
    int tile = xcd_remap(blockIdx.x, gridDim.x);
    if(apart)
        stage(tile);
    __syncthreads();

    // the filter's operands of this wavefront's channels: taps 2g and 2g + 1 of row r, g = hi + 2 * kk
    const int halves_of = (t.K + 31) / 32, j = wave % halves_of;
    half8_t fb[R][2];
#pragma unroll
    for(int r = 0; r < R; r++)
#pragma unroll
        for(int kk = 0; kk < 2; kk++) {
            const int ch = 32 * j + l, tap = 2 * (hi + 2 * kk);
            const bool one = ch < t.K && tap < t.S, two = ch < t.K && tap + 1 < t.S;
            const int at = one ? ((ch * R + r) * t.S + tap) * 6 : 0;
            const unsigned *src = (const unsigned *)(smem + t.w_at + (at & ~3));
            const unsigned d0 = src[0], d1 = src[1], d2 = src[2], d3 = src[3], by = (at & 2) * 8;
            const unsigned e0 = __builtin_amdgcn_alignbit(d1, d0, by), e1 = __builtin_amdgcn_alignbit(d2, d1, by),
                           e2 = __builtin_amdgcn_alignbit(d3, d2, by);
            uint4_t v;
            v[0] = one ? e0 : 0;
            v[1] = one ? e1 & 0xffffu : 0;
            v[2] = two ? __builtin_amdgcn_alignbit(e2, e1, 16) : 0;
            v[3] = two ? e2 >> 16 : 0;
            fb[r][kk] = __builtin_bit_cast(half8_t, v);
        }
    float sc[16], sh[16];
#pragma unroll
    for(int v = 0; v < 16; v++) {
        const int ch = 32 * j + 8 * (v / 4) + 4 * hi + v % 4, c = ch < t.K ? ch : 0;
        sc[v] = t.s[c] * rsqrtf(t.v[c] + t.eps);
        sh[v] = t.b[c] - t.m[c] * sc[v];
    }
    const int run_rows = (t.TP + t.runs - 1) / t.runs;
    if(!apart)
        __syncthreads();
    const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) void *)smem;

    for(; tile < t.ntiles; tile += gridDim.x) {
        if(!apart || tile >= (int)gridDim.x) {
            if(tile >= (int)gridDim.x)
                __syncthreads();
            stage(tile);
            __syncthreads();
        }
        const int n = tile / t.strips, p0 = (tile - n * t.strips) * t.TP, rows = std::min(t.TP, t.Pp - p0);
        for(int item = wave; item < t.items; item += 4) {
            const int rest = item / halves_of, group = rest % t.groups, run = rest / t.groups; // (halves divide four: still half j)
            const int first = run * run_rows, behind = std::min(first + run_rows, rows);
            if(first >= behind)
                continue;
            const int q = 31 * group + l, qe = std::min(q, t.Qp - 1);
            const unsigned at_even = lds0 + hi * t.plane + qe * 16;
            const unsigned at_odd = lds0 + (hi ? (qe + 1) * 16 : t.plane + qe * 16);
            const unsigned keep = 2 * q + 1 < t.Q ? 0xffffffffu : 0u;      // odd columns inside the image
            const unsigned left = group == 0 && l == 0 ? 0u : 0xffffffffu; // there is a column to the left
            auto window = [&](unsigned at, int row, int kk) {
                return __builtin_bit_cast(half8_t, *(lds_vec_t)(uintptr_t)(at + row * t.row + kk * 16));
            };
            auto packed = [&](const float16_t &acc, unsigned (&o)[8]) {
#pragma unroll
                for(int k = 0; k < 8; k++) {
                    half2_t h;
#pragma unroll
                    for(int e = 0; e < 2; e++)
                        h[e] = (half_t)__builtin_elementwise_maximum(__builtin_fmaf(acc[2 * k + e], sc[2 * k + e], sh[2 * k + e]), 0.0f);
                    o[k] = __builtin_bit_cast(unsigned, h);
                }
            };
            unsigned pe[8], po[8]; // the convolution's row above, even and odd columns
#pragma unroll
            for(int k = 0; k < 8; k++)
                pe[k] = po[k] = 0;
            if(p0 + first > 0) {
                float16_t e, o;
#pragma unroll
                for(int v = 0; v < 16; v++)
                    e[v] = o[v] = 0.0f;
#pragma unroll
                for(int r = 0; r < R; r++)
#pragma unroll
                    for(int kk = 0; kk < 2; kk++) {
                        e = __builtin_amdgcn_mfma_f32_32x32x16_f16(fb[r][kk], window(at_even, 4 * first + r, kk), e, 0, 0, 0);
                        o = __builtin_amdgcn_mfma_f32_32x32x16_f16(fb[r][kk], window(at_odd, 4 * first + r, kk), o, 0, 0, 0);
                    }
                packed(e, pe);
                packed(o, po);
            }
            half_t *out = t.y + (((int64_t)n * t.Pp + p0 + first) * t.Qp + q) * t.ldy + 32 * j + 8 * hi;
            const bool store = q < t.Qp && (l > 0 || group == 0);
            for(int p = first; p < behind; p++) {
                float16_t e[2], o[2];
#pragma unroll
                for(int a = 0; a < 2; a++)
#pragma unroll
                    for(int v = 0; v < 16; v++)
                        e[a][v] = o[a][v] = 0.0f;
#pragma unroll
                for(int i = 0; i < R + 2; i++)
#pragma unroll
                    for(int kk = 0; kk < 2; kk++) {
                        const half8_t we = window(at_even, 4 * p + 2 + i, kk), wo = window(at_odd, 4 * p + 2 + i, kk);
                        if(i < R) {
                            e[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fb[i < R ? i : 0][kk], we, e[0], 0, 0, 0);
                            o[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fb[i < R ? i : 0][kk], wo, o[0], 0, 0, 0);
                        }
                        if(i >= 2) {
                            e[1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fb[i >= 2 ? i - 2 : 0][kk], we, e[1], 0, 0, 0);
                            o[1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fb[i >= 2 ? i - 2 : 0][kk], wo, o[1], 0, 0, 0);
                        }
                    }
                unsigned e0[8], o0[8], e1[8], o1[8], w[8];
                packed(e[0], e0);
                packed(o[0], o0);
                packed(e[1], e1);
                packed(o[1], o1);
                const unsigned below = 2 * (p0 + p) + 1 < t.P ? 0xffffffffu : 0u;
#pragma unroll
                for(int k = 0; k < 8; k++) {
                    e1[k] &= below;
                    o1[k] &= below;
                    const unsigned even = largest(pe[k], e0[k], e1[k]), odd = largest(po[k], o0[k], o1[k]) & keep;
                    const unsigned before = __builtin_amdgcn_update_dpp(0, odd, 0x138, 0xf, 0xf, true) & left; // wave_shr:1
                    w[k] = largest(even, odd, before);
                    pe[k] = e1[k];
                    po[k] = o1[k];
                }
                // channels 16k .. 16k + 7 of the pixel to the lower half of the wavefront, the next eight to the upper
#pragma unroll
                for(int k = 0; k < 2; k++) {
                    const auto s0 = __builtin_amdgcn_permlane32_swap(w[4 * k], w[4 * k + 2], false, false);
                    const auto s1 = __builtin_amdgcn_permlane32_swap(w[4 * k + 1], w[4 * k + 3], false, false);
                    const uint4_t v = {s0[0], s1[0], s0[1], s1[1]};
                    if(store && 32 * j + 16 * k + 8 * hi < t.K)
                        *(uint4_t *)(out + 16 * k) = v;
                }
                out += (int64_t)t.Qp * t.ldy;
            }
        }
    }
}

constexpr int MAX_LDS = 80 * 1024 - 256; // of two blocks on a CU

// the launch, or ntiles 0: not this kernel's
StemArgs plan(const SagaTensorView *x, const SagaTensorView *w, const SagaTensorView *y, const ConvGeom &g, int size, int pool_pad,
              int pool_stride)
{
    StemArgs t = {};
    CLInfo lx, lw, ly;
    if(x->dtype != SAGA_HALF || w->dtype != SAGA_HALF || y->dtype != SAGA_HALF || size != 3 || pool_stride != 2 || pool_pad != 1 ||
       g.R != R || g.S > 8 || g.C != 3 || g.stride != 2 || g.dil != 1 || g.group != 1 || g.pad > 3 || g.K > 64 || g.K % 8 ||
       !as_channels_last(x, &lx) || !as_channels_last(w, &lw) || !as_channels_last(y, &ly) || lx.pitch != 3 || lw.pitch != 3 || ly.pitch % 8)
        return t;
    t.H = g.H, t.W = g.W, t.P = g.P, t.Q = g.Q, t.K = g.K, t.S = g.S, t.pad = g.pad;
    t.Pp = (g.P - 1) / 2 + 1;
    t.Qp = (g.Q - 1) / 2 + 1;
    if(y->dims[0] != g.N || y->dims[1] != g.K || y->dims[2] != t.Pp || y->dims[3] != t.Qp)
        return t;
    const int64_t image = (int64_t)g.H * g.W * 6;
    if(image >= 0x7fff0000 || (int64_t)g.N * t.Pp >= 0x7fffffff)
        return t;
    t.x_bytes = (int)image;
    t.ldy = ly.pitch;
    t.pieces = 2 * (t.Qp + 2);
    t.plane = (t.Qp + 2) * 16;
    t.row = 2 * t.plane;
    t.w_bytes = g.K * R * g.S * 6;
    t.groups = t.Qp <= 32 ? 1 : 1 + (t.Qp - 32 + 30) / 31;
    const int halves_of = (g.K + 31) / 32;
    // Pooled rows of a strip: what makes the least of the rounds that the blocks go, two on a CU, each a staging, the row above
    // again and the rows.
    const int64_t slots = 512;
    int64_t least = 0;
    for(int tp = 1; tp <= 16 && (4 * tp + R) * t.row <= MAX_LDS; tp++)
        for(int runs = 1; runs <= 4 && runs <= tp; runs *= 2) {
            const int strips = (t.Pp + tp - 1) / tp;
            const int64_t rounds = ((int64_t)g.N * strips + slots - 1) / slots;
            const int items = halves_of * t.groups * runs, turns = (items + 3) / 4, rows = (tp + runs - 1) / runs;
            const int64_t cost = rounds * (turns * (2 * rows + 1) * 4 + 4 * tp + R);
            if(!least || cost < least) {
                least = cost;
                t.TP = tp;
                t.runs = runs;
                t.strips = strips;
                t.items = items;
                t.ntiles = g.N * strips;
            }
        }
    return t;
}

} // namespace

bool conv_bn_maxpool_ok(const SagaTensorView *x, const SagaTensorView *w, const SagaTensorView *y, const ConvGeom &g, int size,
                        int pool_pad, int pool_stride)
{
    return aligned16(w->ptr) && aligned16(y->ptr) && plan(x, w, y, g, size, pool_pad, pool_stride).ntiles > 0;
}

int conv_bn_maxpool(const SagaTensorView *x, const SagaTensorView *w, const SagaTensorView *y, const ConvGeom &g, const float *s,
                    const float *b, const float *m, const float *v, float eps, int size, int pool_pad, int pool_stride, hipStream_t st)
{
    if(!conv_bn_maxpool_ok(x, w, y, g, size, pool_pad, pool_stride))
        return SAGA_HIP_EUNSUPPORTED;
    StemArgs t = plan(x, w, y, g, size, pool_pad, pool_stride);
    t.x = (const half_t *)x->ptr;
    t.w = (const half_t *)w->ptr;
    t.y = (half_t *)y->ptr;
    t.s = s, t.b = b, t.m = m, t.v = v;
    t.eps = eps;
    const int rows = (4 * t.TP + R) * t.row, filter = t.w_bytes + 16;
    t.w_at = rows + filter <= MAX_LDS ? rows : 0;
    const int lds = t.w_at ? rows + filter : std::max(rows, filter);
    static const hipError_t allowed = hipFuncSetAttribute((const void *)conv7x7s2_bn_maxpool, hipFuncAttributeMaxDynamicSharedMemorySize, MAX_LDS);
    if(allowed != hipSuccess)
        return (int)allowed;
    conv7x7s2_bn_maxpool<<<std::min(t.ntiles, 512), 256, lds, st>>>(t);
    SAGA_CHECK_LAUNCH();
    return 0;
}
