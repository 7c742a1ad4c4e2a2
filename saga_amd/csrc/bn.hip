// Batch normalisation for gfx950: inference, training forward (with optional fused
// residual add + relu) and backward.  Everything here is HBM-bound.
//
// Channels-last tensors are walked as rows of C contiguous channels: a 256-thread block is
// shaped (CVB channel-vectors) x (RB rows); lanes along x read consecutive 16-byte vectors so
// each wavefront touches whole rows, and every thread keeps its channel's parameters in
// registers for all the rows it visits.  Per-channel sums are reduced thread -> LDS ->
// per-block partials in the workspace -> one small finalize kernel, so the data is read
// exactly twice in training forward (statistics, then normalise) and backward.
//
// Statistics are accumulated on values shifted by the channel's first element, which removes
// the cancellation in E[x^2] - E[x]^2 when |mean| >> stddev.
#include "common.hpp"

#include <stdlib.h>

#include <algorithm>

namespace {

template <typename T, int VN> struct VecT;
template <> struct VecT<half_t, 8> { typedef half8_t type; };
template <> struct VecT<float, 4> { typedef float4_t type; };
template <> struct VecT<half_t, 1> { typedef half_t type; };
template <> struct VecT<float, 1> { typedef float type; };

template <typename T, int VN, bool NT = true> struct Ld {
    typedef typename VecT<T, VN>::type V;
    static __device__ __forceinline__ void load(const T *p, float (&o)[VN])
    {
        if constexpr(VN == 1) {
            o[0] = (float)*p;
        } else {
            // (non-temporal, like the stores below: these kernels read every tensor once; 9.18 -> 8.99 ms for the
            // batch-norm kernels of a ResNet-50 training step)
            const V v = NT ? __builtin_nontemporal_load((const V *)p) : *(const V *)p;
#pragma unroll
            for(int j = 0; j < VN; j++)
                o[j] = (float)v[j];
        }
    }
    static __device__ __forceinline__ V raw(const T *p) { return NT ? __builtin_nontemporal_load((const V *)p) : *(const V *)p; }
    static __device__ __forceinline__ float at(const V &v, int j)
    {
        if constexpr(VN == 1)
            return (float)v;
        else
            return (float)v[j];
    }
    static __device__ __forceinline__ void store(T *p, const float (&o)[VN])
    {
        if constexpr(VN == 1) {
            *p = (T)o[0];
        } else {
            V v;
#pragma unroll
            for(int j = 0; j < VN; j++)
                v[j] = (T)o[j];
            // non-temporal: what these kernels write is a stream that the next operation reads whole; with the hint
            // the batch-norm kernels of a ResNet-50 training step take 9.06 ms instead of 9.23, and the convolutions
            // that read the results take what they took
            __builtin_nontemporal_store(v, (V *)p);
        }
    }
};

struct Shape {
    int cvb;  // channel vectors per block (power of two <= 64)
    int rb;   // rows per block = 256 / cvb
    int gy;   // blocks along channels
    int gx;   // blocks along rows of the kernels that leave one partial row per block
    int gxa;  // blocks along rows of the kernels that only stream (no partials: as many as there are batches)
};

static int env_int(const char *name, int dflt)
{
    const char *e = getenv(name);
    return e && *e ? atoi(e) : dflt;
}

// backward: the statistics pass leaves fewer partial rows (measured on MI355X inside the ResNet-50 step: 512
// blocks of contiguous row runs beat 2048 by 3 %), and the apply pass that follows uses the same small grid
static Shape plan(int64_t rows, int cvec, bool backward = false)
{
    Shape s;
    s.cvb = 1;
    while(s.cvb < cvec && s.cvb < 64)
        s.cvb <<= 1;
    s.rb = 256 / s.cvb;
    s.gy = (cvec + s.cvb - 1) / s.cvb;
    // SAGA_HIP_BN_STATS_BLOCKS / SAGA_HIP_BN_APPLY_GROUPS: experiment knobs (blocks of a reducing kernel over the
    // whole tensor; row groups per block of a streaming kernel)
    static const int fwd_blocks = env_int("SAGA_HIP_BN_STATS_BLOCKS", 2048);
    static const int bwd_blocks = env_int("SAGA_HIP_BN_BWD_BLOCKS", 512);
    const int stats_blocks = backward ? bwd_blocks : fwd_blocks;
    static const int apply_groups = env_int("SAGA_HIP_BN_APPLY_GROUPS", 4);
    int64_t want = (rows + (int64_t)s.rb * 4 - 1) / ((int64_t)s.rb * 4);
    int cap = stats_blocks / s.gy;
    if(cap < 1)
        cap = 1;
    if(want > cap)
        want = cap;
    if(want < 1)
        want = 1;
    s.gx = (int)want;
    int64_t wa = (rows + (int64_t)s.rb * apply_groups - 1) / ((int64_t)s.rb * apply_groups);
    if(wa > 65535)
        wa = 65535;
    if(wa < 1)
        wa = 1;
    s.gxa = (int)wa;
    return s;
}

// ---------------------------------------------------------------- channels-last kernels

// Rows of a block.  Either a block owns a CONTIGUOUS run of row groups (rb rows each) and walks it in order, so
// that the batch of rows it has in flight is one contiguous piece of memory and the blocks, dispatched in order,
// sweep the tensor front to back; or (cvb < 0) the grid-stride walk, where the rows of a batch lie a whole grid
// apart.  On tensors that come from HBM the first order is much faster (a plain copy moves 5.4 - 6 TB/s that way
// and 4.1 - 4.5 TB/s grid-strided; batch-norm backward on 411 MB tensors 367 us against 494 us).  Inside a
// training step part of the data is still in the last-level cache and the picture is mixed - measured per kernel
// on the ResNet-50 b256 step: the backward statistics pass gains 5 % from contiguous runs with 512 blocks, the
// two apply passes lose 2 - 7 % - hence the default of gridstride_mask().  r0 = first row of this thread,
// rend = end of the block's run, stride = distance of a thread's consecutive rows.
struct RowRun {
    int64_t r0, rend, stride;
};
__device__ __forceinline__ RowRun row_run(int64_t rows, int rb, int ty, int cvb)
{
    RowRun rr;
    if(cvb < 0) {
        rr.r0 = (int64_t)blockIdx.x * rb + ty;
        rr.rend = rows;
        rr.stride = (int64_t)gridDim.x * rb;
        return rr;
    }
    const int64_t groups = (rows + rb - 1) / rb;
    const int64_t per = (groups + gridDim.x - 1) / gridDim.x;
    const int64_t g0 = (int64_t)blockIdx.x * per;
    int64_t g1 = g0 + per;
    if(g1 > groups)
        g1 = groups;
    rr.r0 = g0 * rb + ty;
    rr.rend = g1 * rb < rows ? g1 * rb : rows;
    rr.stride = rb;
    return rr;
}

// Small tensors: the streaming pass finalizes the statistics itself.  A launch that does nothing but add partial sums costs
// 3 - 5 us and the pause in front of the next; here every block adds the partials of its slab of up to 64 channels again,
// while its first rows are on their way (us of finalizing and normalizing, before -> after: 64 channels of 128x8x8 from 32
// partial rows 6.8 -> 4.7, 1024 of 23x13x13 from 16 11.0 -> 7.0).  The blocks of row 0 write what outlives the launch.  Where there are
// thousands of partials or blocks, reading them again costs more than the launch (see self_finalizing).
struct StatsFin {
    const float *partial;
    int prows;
    const float *s, *b;
    float *run_m, *run_v, *save_mean, *save_invstd;
    double M;
    float eps, expavg;
};
struct BwdFin {
    const float *partial;
    int prows;
    const float *s, *save_invstd;
    float *ds, *db;
    double M;
    float beta_p;
};

// Every `lanes`-th of the partials from row l on, up to N of them, which are all on their way at once.
template <int N> __device__ __forceinline__ void lane_sums(const float *__restrict__ partial, int prows, int C, int c, int l, int lanes, double &a0, double &a1)
{
    typedef float float2_t __attribute__((ext_vector_type(2)));
    const float2_t *p = (const float2_t *)partial + c;
    float2_t v[N];
#pragma unroll
    for(int u = 0; u < N; u++)
        v[u] = p[(int64_t)(l + u * lanes < prows ? l + u * lanes : 0) * C];
#pragma unroll
    for(int u = 0; u < N; u++)
        if(l + u * lanes < prows) {
            a0 += v[u][0];
            a1 += v[u][1];
        }
}

// totals of a slab of CS channels from cb on: valid for threads below CS.  A thread's partials (32 at most, MOST backward) are one trip to
// memory: in batches of eight, one after the other, normalizing 16 channels of 128x32x32 from 512 rows took 9.6 us and now takes 7.7,
// the backward of 32 of 128x16x16 7.8 and 7.2; and no more loads than needed, 1024 of 23x13x13 from 61 rows 7.2 with 8, 9.1 with 32.
template <int MOST>
__device__ __forceinline__ void slab_sums(const float *__restrict__ partial, int prows, int C, int cb, int CS, double &s0, double &s1)
{
    __shared__ double red[2][256];
    const int tid = threadIdx.x, c = cb + tid % CS < C ? cb + tid % CS : 0, l = tid / CS, lanes = 256 / CS;
    double a0 = 0, a1 = 0;
    int g = l;
    if(MOST > 16 && prows > 16 * lanes)
        for(; g < prows; g += MOST * lanes)
            lane_sums<MOST>(partial, prows, C, c, g, lanes, a0, a1);
    else if(prows > 8 * lanes)
        for(; g < prows; g += 16 * lanes)
            lane_sums<16>(partial, prows, C, c, g, lanes, a0, a1);
    else
        lane_sums<8>(partial, prows, C, c, g, lanes, a0, a1);
    red[0][tid] = a0;
    red[1][tid] = a1;
    __syncthreads();
    s0 = s1 = 0;
    if(tid < CS)
        for(int k = 0; k < lanes; k++) {
            s0 += red[0][k * CS + tid];
            s1 += red[1][k * CS + tid];
        }
}

// mean, biased variance, 1/std and what follows from them, as bn_stats_finalize has it
__device__ __forceinline__ void finish_stats(double s0, double s1, double k, double M, float eps, float expavg, float sv, float bv,
                                             float rm_old, float rv_old, bool write, float *run_m, float *run_v, float *save_mean,
                                             float *save_invstd, int c, float &scale, float &shift)
{
    const double dm = s0 / M;
    double var = s1 / M - dm * dm;
    if(var < 0)
        var = 0;
    const double mean = k + dm;
    const float inv = (float)(1.0 / sqrt(var + (double)eps));
    if(write) {
        if(save_mean)
            save_mean[c] = (float)mean;
        if(save_invstd)
            save_invstd[c] = inv;
        if(run_m)
            run_m[c] = (float)((1.0 - expavg) * rm_old + expavg * mean);
        if(run_v) {
            const double unb = M > 1 ? var * M / (M - 1.0) : var;
            run_v[c] = (float)((1.0 - expavg) * rv_old + expavg * unb);
        }
    }
    scale = sv * inv;
    shift = __builtin_fmaf(-(float)mean, scale, bv); // same expression as the backward mask recompute
}

__device__ __forceinline__ void stats_slab(const StatsFin &f, int C, int cb, int CS, float (&tab)[2][64])
{
    const int tid = threadIdx.x, c = cb + tid;
    const bool own = tid < CS && c < C, write = blockIdx.x == 0;
    float sv = 0, bv = 0, rm = 0, rv = 0;
    if(own) {
        sv = f.s[c];
        bv = f.b[c];
        if(write && f.run_m)
            rm = f.run_m[c];
        if(write && f.run_v)
            rv = f.run_v[c];
    }
    double s0, s1;
    slab_sums<32>(f.partial, f.prows, C, cb, CS, s0, s1);
    if(own)
        finish_stats(s0, s1, 0.0, f.M, f.eps, f.expavg, sv, bv, rm, rv, write, f.run_m, f.run_v, f.save_mean, f.save_invstd, c,
                     tab[0][tid], tab[1][tid]);
    __syncthreads();
}

__device__ __forceinline__ void bwd_slab(const BwdFin &f, int C, int cb, int CS, float (&tab)[3][64])
{
    const int tid = threadIdx.x, c = cb + tid;
    const bool own = tid < CS && c < C, write = blockIdx.x == 0;
    float sv = 0, inv = 0, ds_old = 0, db_old = 0;
    if(own) {
        sv = f.s[c];
        inv = f.save_invstd[c];
        if(write && f.beta_p != 0.0f) {
            ds_old = f.ds[c];
            db_old = f.db[c];
        }
    }
    double s0, s1;
    slab_sums<16>(f.partial, f.prows, C, cb, CS, s0, s1);
    if(own) {
        const double dsv = s1 * inv;
        if(write) {
            f.ds[c] = (float)(f.beta_p != 0.0f ? dsv + (double)f.beta_p * ds_old : dsv);
            f.db[c] = (float)(f.beta_p != 0.0f ? s0 + (double)f.beta_p * db_old : s0);
        }
        tab[0][tid] = (float)(sv * (double)inv);
        tab[1][tid] = (float)(s0 / f.M);
        tab[2][tid] = (float)(dsv * inv / f.M);
    }
    __syncthreads();
}

// Grid of a self-finalizing pass (blocks of four row groups, about a thousand at most), or false.  A thread adds at most 32
// partials forward (128 rows of 64 channels, 512 of 16) and 16 backward, where its registers leave fewer wavefronts to hide
// that (us, separate / own finalizing: forward 512 channels of 23x25x25 11.1 / 9.5;
// linked backward of 1024 of 23x13x13 10.3 / 8.0, 512 of 23x25x25 13 / 15, 16 of 128x32x32 from 512
// rows 7.0 / 8.5).
static bool self_finalizing(int64_t rows, int C, int prows, bool backward, Shape *sh)
{
    const int cvec = C / 8;
    int cvb = 1;
    while(cvb < cvec && cvb < 8)
        cvb <<= 1;
    const int rb = 256 / cvb, lanes = 256 / (cvb * 8);
    if(C % 8 || prows > (backward ? 16 : 32) * lanes)
        return false;
    sh->cvb = cvb;
    sh->rb = rb;
    sh->gy = (cvec + cvb - 1) / cvb;
    const int64_t groups = (rows + rb - 1) / rb;
    if(groups * sh->gy > (backward ? 2400 : 4096))
        return false;
    sh->gx = sh->gxa = (int)((groups + 3) / 4);
    return true;
}

// y = x*scale[c] + shift[c] (+ z) (relu).  MODE 0: scale/shift from s,b,m,v (inference);
// MODE 1: scale/shift precomputed in ss[0..C), ss[C..2C) (training, second pass); MODE 2: from partial sums (StatsFin).
template <typename T, int VN, int MODE>
__global__ void __launch_bounds__(256)
    bn_apply_cl(const T *__restrict__ x, int64_t px, const T *__restrict__ z, int64_t pz, T *__restrict__ y, int64_t py,
                const float *__restrict__ s, const float *__restrict__ b, const float *__restrict__ m,
                const float *__restrict__ v, const float *__restrict__ ss, float eps, int64_t rows, int C, int cvb_,
                int flags, uint8_t *__restrict__ mask = nullptr, StatsFin fin = StatsFin())
{
    // mask (VN == 8 only): one byte per row and 8-channel vector, bit j set where the stored y is > 0;
    // the backward pass of a fused add + relu layer reads it instead of y
    const int cvb = cvb_ < 0 ? -cvb_ : cvb_;
    const int tx = threadIdx.x % cvb, ty = threadIdx.x / cvb, rb = 256 / cvb;
    const int c0 = (blockIdx.y * cvb + tx) * VN;
    if(MODE != 2 && c0 >= C)
        return;
    float sc[VN], sh[VN];
#pragma unroll
    for(int j = 0; j < VN; j++) {
        if(MODE == 0) {
            sc[j] = s[c0 + j] * rsqrtf(v[c0 + j] + eps);
            sh[j] = b[c0 + j] - m[c0 + j] * sc[j];
        } else if(MODE == 1) {
            sc[j] = ss[c0 + j];
            sh[j] = ss[C + c0 + j];
        }
    }
    const bool relu = flags & SAGA_BN_RELU, add = flags & SAGA_BN_ADD;
    typedef Ld<T, VN> L;
    typedef typename L::V V;
    // MODE 1 and 2 run right after the statistics pass over the same rows: walking them in the
    // opposite direction meets the rows that pass touched last, which are the ones most
    // likely to be still cached
    const RowRun rr = row_run(rows, rb, ty, cvb_);
    const int64_t stride = rr.stride;
    auto row = [&](int64_t r) { return MODE >= 1 ? rows - 1 - r : r; };
    auto finish = [&](const V &xr, const V &zr, int64_t r) {
        float o[VN];
#pragma unroll
        for(int j = 0; j < VN; j++) {
            float t = __builtin_fmaf(L::at(xr, j), sc[j], sh[j]);
            if(add)
                t += L::at(zr, j);
            if(relu)
                t = (t != t) ? t : fmaxf(t, 0.0f);
            o[j] = t;
        }
        L::store(y + r * py + c0, o);
        if constexpr(VN == 8) {
            if(mask) {
                unsigned bits = 0;
#pragma unroll
                for(int j = 0; j < VN; j++)
                    bits |= ((float)(T)o[j] > 0.0f ? 1u : 0u) << j;
                __builtin_nontemporal_store((uint8_t)bits, mask + r * (C / VN) + c0 / VN); // (read again in the backward pass only)
            }
        }
    };
    int64_t r = rr.r0;
    const int64_t rend = rr.rend;
    V xr[4], zr[4];
    auto load4 = [&]() {
#pragma unroll
        for(int u = 0; u < 4; u++) {
            xr[u] = L::raw(x + row(r + u * stride) * px + c0);
            zr[u] = add ? L::raw(z + row(r + u * stride) * pz + c0) : xr[u];
        }
    };
    auto finish4 = [&]() {
#pragma unroll
        for(int u = 0; u < 4; u++)
            finish(xr[u], zr[u], row(r + u * stride));
        r += 4 * stride;
    };
    if constexpr(MODE == 2) {
        __shared__ float tab[2][64];
        const bool ahead = c0 < C && r + 3 * stride < rend;
        if(ahead)
            load4();
        stats_slab(fin, C, blockIdx.y * cvb * VN, cvb * VN, tab);
        if(c0 >= C)
            return;
#pragma unroll
        for(int j = 0; j < VN; j++) {
            sc[j] = tab[0][tx * VN + j];
            sh[j] = tab[1][tx * VN + j];
        }
        if(ahead)
            finish4();
    }
    while(r + 3 * stride < rend) {
        load4();
        finish4();
    }
    for(; r < rend; r += stride) {
        const V xr = L::raw(x + row(r) * px + c0);
        const V zr = add ? L::raw(z + row(r) * pz + c0) : xr;
        finish(xr, zr, row(r));
    }
}

// The sums of a block's 256 / cvb row lanes, for its cvb channel vectors, into its row of partials.  All threads take part,
// in a fixed order (one row of threads that walked the others' values took 4 us of the 10 that the backward statistics of
// 16 channels need).  red: (256 + cvb) * 2 * VN floats; the pitch keeps the walks off each other's banks.
template <int VN>
__device__ __forceinline__ void block_partials(const float (&a0)[VN], const float (&a1)[VN], float *red, int tx, int cvb,
                                               float *__restrict__ partial, int C)
{
    const int tid = threadIdx.x, pitch = 256 + cvb, rb = 256 / cvb, sums = cvb * 2 * VN;
#pragma unroll
    for(int j = 0; j < VN; j++) {
        red[j * pitch + tid] = a0[j];
        red[(VN + j) * pitch + tid] = a1[j];
    }
    __syncthreads();
    const int parts = sums < 256 ? 256 / sums : 1; // threads per sum
    const int len = (rb + parts - 1) / parts;
    float *o = partial + ((int64_t)blockIdx.x * C + blockIdx.y * cvb * VN) * 2;
    auto store = [&](int q, float v) {
        const int k = q / cvb, c = (q % cvb) * VN + k % VN; // k: the value's number in its thread
        if((int)blockIdx.y * cvb * VN + c < C)
            o[c * 2 + k / VN] = v;
    };
    if(parts == 1) { // few rows: one of them adds the others
        const int c0 = (blockIdx.y * cvb + tx) * VN;
        if(tid >= cvb || c0 >= C)
            return;
        float t0[VN], t1[VN];
#pragma unroll
        for(int j = 0; j < VN; j++) {
            t0[j] = a0[j];
            t1[j] = a1[j];
        }
        for(int t = 1; t < rb; t++)
#pragma unroll
            for(int j = 0; j < VN; j++) {
                t0[j] += red[j * pitch + t * cvb + tx];
                t1[j] += red[(VN + j) * pitch + t * cvb + tx];
            }
#pragma unroll
        for(int j = 0; j < VN; j++) {
            o[(tx * VN + j) * 2] = t0[j];
            o[(tx * VN + j) * 2 + 1] = t1[j];
        }
        return;
    }
    const int q = tid % sums, p = tid / sums;
    float v = 0;
    for(int t = p * len; t < (p + 1) * len && t < rb; t++)
        v += red[(q / cvb) * pitch + t * cvb + q % cvb];
    __syncthreads();
    red[tid] = v;
    __syncthreads();
    if(tid < sums) {
        for(int k = 1; k < parts; k++)
            v += red[k * sums + tid];
        store(tid, v);
    }
}

// Pass 1 of training forward: per-block partial sums of (x-K) and (x-K)^2, K = x[row 0].
template <typename T, int VN>
__global__ void __launch_bounds__(256)
    bn_stats_cl(const T *__restrict__ x, int64_t px, float *__restrict__ partial, int64_t rows, int C, int cvb_)
{
    __shared__ float red[320 * VN * 2];
    const int cvb = cvb_ < 0 ? -cvb_ : cvb_;
    const int tx = threadIdx.x % cvb, ty = threadIdx.x / cvb, rb = 256 / cvb;
    const int c0 = (blockIdx.y * cvb + tx) * VN;
    float a0[VN], a1[VN], k[VN];
#pragma unroll
    for(int j = 0; j < VN; j++)
        a0[j] = a1[j] = 0.0f;
    if(c0 < C) {
        typedef Ld<T, VN, false> L;
        typedef typename L::V V;
        L::load(x + c0, k);
        const RowRun rr = row_run(rows, rb, ty, cvb_);
        const int64_t stride = rr.stride;
        const int64_t rend = rr.rend;
        auto add = [&](const V &xr) {
#pragma unroll
            for(int j = 0; j < VN; j++) {
                const float d = L::at(xr, j) - k[j];
                a0[j] += d;
                a1[j] += d * d;
            }
        };
        int64_t r = rr.r0;
        for(; r + 7 * stride < rend; r += 8 * stride) {
            V xr[8];
#pragma unroll
            for(int u = 0; u < 8; u++)
                xr[u] = L::raw(x + (r + u * stride) * px + c0);
#pragma unroll
            for(int u = 0; u < 8; u++)
                add(xr[u]);
        }
        for(; r < rend; r += stride)
            add(L::raw(x + r * px + c0));
    }
    block_partials<VN>(a0, a1, red, tx, cvb, partial, C);
}

__device__ __forceinline__ double wave_sum_f64(double v)
{
#pragma unroll
    for(int o = 32; o > 0; o >>= 1)
        v += __shfl_xor(v, o, 64);
    return v;
}

// Adds the gx per-block partial pairs of channel c over the four wavefronts of a block, in a
// fixed order.  The loads of a thread are independent: eight are issued before any is consumed,
// and with 256 threads on one channel even 2048 partials are one such batch per thread, so the
// block pays the memory latency about once (these kernels are nothing but latency).
// The totals are valid in thread 0 only.
__device__ __forceinline__ void sum_partials(const float *__restrict__ partial, int gx, int C, int c, double &s0,
                                             double &s1)
{
    typedef float float2_t __attribute__((ext_vector_type(2)));
    __shared__ double red[4][2];
    const float2_t *p = (const float2_t *)partial + c;
    const int tid = threadIdx.x;
    double a0 = 0, a1 = 0;
    int g = tid;
    for(; g + 7 * 256 < gx; g += 8 * 256) {
        float2_t v[8];
#pragma unroll
        for(int u = 0; u < 8; u++)
            v[u] = p[(int64_t)(g + u * 256) * C];
#pragma unroll
        for(int u = 0; u < 8; u++) {
            a0 += v[u][0];
            a1 += v[u][1];
        }
    }
    {
        // the remainder, again as one batch: out-of-range slots read row 0 and are not added
        float2_t v[8];
#pragma unroll
        for(int u = 0; u < 8; u++) {
            const int r = g + u * 256;
            v[u] = p[(int64_t)(r < gx ? r : 0) * C];
        }
#pragma unroll
        for(int u = 0; u < 8; u++)
            if(g + u * 256 < gx) {
                a0 += v[u][0];
                a1 += v[u][1];
            }
    }
    a0 = wave_sum_f64(a0);
    a1 = wave_sum_f64(a1);
    if((tid & 63) == 0) {
        red[tid >> 6][0] = a0;
        red[tid >> 6][1] = a1;
    }
    __syncthreads();
    s0 = red[0][0] + red[1][0] + red[2][0] + red[3][0];
    s1 = red[0][1] + red[1][1] + red[2][1] + red[3][1];
}

// Finalize: mean, biased variance, invstd, running statistics, fused scale/shift.
// One block per channel adds the per-block partials (threads stride over the blocks).
template <typename T>
__global__ void __launch_bounds__(256)
    bn_stats_finalize(const float *__restrict__ partial, int gx, const T *__restrict__ xrow0, int64_t kstride,
                      const float *__restrict__ s, const float *__restrict__ b, float *run_m, float *run_v,
                      float *save_mean, float *save_invstd, float *ss, double M, int C, float eps, float expavg)
{
    const int c = blockIdx.x;
    // parameter loads first: they overlap the partial-sum loads instead of following them
    const double k = xrow0 ? (double)(float)xrow0[c * kstride] : 0.0;
    const float sv = s[c], bv = b[c];
    const float rm_old = run_m ? run_m[c] : 0.0f, rv_old = run_v ? run_v[c] : 0.0f;
    double s0, s1;
    sum_partials(partial, gx, C, c, s0, s1);
    if(threadIdx.x != 0)
        return;
    finish_stats(s0, s1, k, M, eps, expavg, sv, bv, rm_old, rv_old, true, run_m, run_v, save_mean, save_invstd, c, ss[c], ss[C + c]);
}

// Pass 1 of backward: partial sums of dy' and dy'*(x-mean); dy' = dy masked by y>0 when fused relu.
template <typename T, int VN, bool RC>
__global__ void __launch_bounds__(256)
    bn_bwd_stats_cl(const T *__restrict__ x, int64_t px, const T *__restrict__ y, int64_t py, const T *__restrict__ dy,
                    int64_t pdy, const float *__restrict__ save_mean, float *__restrict__ partial, int64_t rows, int C,
                    int cvb_, int flags, const float *__restrict__ rs, const float *__restrict__ rb_, const float *__restrict__ rinv,
                    T *__restrict__ dz, int64_t pdz, const uint8_t *__restrict__ mask = nullptr)
{
    // mask set (VN == 8): the relu mask comes from the byte per row and channel vector that the
    // forward pass left, and y is not read
    // dz set: the masked gradient dy' is stored there on the way (it is the residual branch's
    // gradient anyway), and the second pass reads it instead of y and dy
    // rs/rb_/rinv (scale, bias, saved 1/std) set: the relu mask is recomputed from x as
    // half(fma(x, sc, sh)) > 0, exactly what the forward stored, and y is not read
    __shared__ float red[320 * VN * 2];
    const int cvb = cvb_ < 0 ? -cvb_ : cvb_;
    const int tx = threadIdx.x % cvb, ty = threadIdx.x / cvb, rb = 256 / cvb;
    const int c0 = (blockIdx.y * cvb + tx) * VN;
    const bool relu = flags & SAGA_BN_RELU;
    constexpr bool recompute = RC;
    float a0[VN], a1[VN], mean[VN], sc[VN], sh[VN];
#pragma unroll
    for(int j = 0; j < VN; j++)
        a0[j] = a1[j] = 0.0f;
    if(c0 < C) {
#pragma unroll
        for(int j = 0; j < VN; j++) {
            mean[j] = save_mean[c0 + j];
            sc[j] = recompute ? rs[c0 + j] * rinv[c0 + j] : 0.0f;
            sh[j] = recompute ? __builtin_fmaf(-mean[j], sc[j], rb_[c0 + j]) : 0.0f;
        }
        typedef Ld<T, VN, false> L;
        typedef typename L::V V;
        const RowRun rr = row_run(rows, rb, ty, cvb_);
        const int64_t stride = rr.stride;
        const int64_t rend = rr.rend;
        auto add = [&](const V &xr, const V &gr, const V &yr, unsigned mb, int64_t r) {
            float gm[VN];
#pragma unroll
            for(int j = 0; j < VN; j++) {
                float g = L::at(gr, j);
                const float yv = recompute ? (float)(T)__builtin_fmaf(L::at(xr, j), sc[j], sh[j])
                                 : mask    ? (float)((mb >> j) & 1u)
                                           : L::at(yr, j);
                if(relu && !(yv > 0.0f))
                    g = 0.0f;
                a0[j] += g;
                a1[j] += g * (L::at(xr, j) - mean[j]);
                gm[j] = g;
            }
            if(dz)
                L::store(dz + r * pdz + c0, gm);
        };
        int64_t r = rr.r0;
        const int mp = C / VN, mc = c0 / VN; // mask row pitch and this thread's byte
        for(; r + 3 * stride < rend; r += 4 * stride) {
            V xr[4], gr[4], yr[4];
            unsigned mb[4];
#pragma unroll
            for(int u = 0; u < 4; u++) {
                xr[u] = L::raw(x + (r + u * stride) * px + c0);
                gr[u] = L::raw(dy + (r + u * stride) * pdy + c0);
                yr[u] = relu && !recompute && !mask ? L::raw(y + (r + u * stride) * py + c0) : gr[u];
                mb[u] = mask ? mask[(r + u * stride) * mp + mc] : 0u;
            }
#pragma unroll
            for(int u = 0; u < 4; u++)
                add(xr[u], gr[u], yr[u], mb[u], r + u * stride);
        }
        for(; r < rend; r += stride) {
            const V xr = L::raw(x + r * px + c0), gr = L::raw(dy + r * pdy + c0);
            add(xr, gr, relu && !recompute && !mask ? L::raw(y + r * py + c0) : gr, mask ? mask[r * mp + mc] : 0u, r);
        }
    }
    block_partials<VN>(a0, a1, red, tx, cvb, partial, C);
}

// coef[0..C) = s*invstd ; coef[C..2C) = db/M ; coef[2C..3C) = ds*invstd/M ; writes ds, db.
// One block per channel, as above.
__global__ void __launch_bounds__(256)
    bn_bwd_finalize(const float *__restrict__ partial, int gx, const float *__restrict__ s,
                    const float *__restrict__ save_invstd, float *ds, float *db, float *coef, double M, int C,
                    float beta_p)
{
    const int c = blockIdx.x;
    const double inv = save_invstd[c];
    const float sv = s[c];
    const float ds_old = beta_p != 0.0f ? ds[c] : 0.0f, db_old = beta_p != 0.0f ? db[c] : 0.0f;
    double s0, s1;
    sum_partials(partial, gx, C, c, s0, s1);
    if(threadIdx.x != 0)
        return;
    const double dsv = s1 * inv;
    ds[c] = (float)(beta_p != 0.0f ? dsv + (double)beta_p * ds_old : dsv);
    db[c] = (float)(beta_p != 0.0f ? s0 + (double)beta_p * db_old : s0);
    coef[c] = (float)(sv * inv);
    coef[C + c] = (float)(s0 / M);
    coef[2 * C + c] = (float)(dsv * inv / M);
}

// Pass 2 of backward: dx = s*invstd*(dy' - db/M - (x-mean)*invstd*ds/M) ; dz = dy'.
template <typename T, int VN, bool RC, bool FIN = false>
__global__ void __launch_bounds__(256)
    bn_bwd_apply_cl(const T *__restrict__ x, int64_t px, const T *__restrict__ y, int64_t py, const T *__restrict__ dy,
                    int64_t pdy, T *__restrict__ dx, int64_t pdx, T *__restrict__ dz, int64_t pdz,
                    const float *__restrict__ save_mean, const float *__restrict__ coef, int64_t rows, int C, int cvb_,
                    int flags, float beta_dx, float beta_dz, const float *__restrict__ rb_, BwdFin fin = BwdFin())
{
    const int cvb = cvb_ < 0 ? -cvb_ : cvb_;
    const int tx = threadIdx.x % cvb, ty = threadIdx.x / cvb, rb = 256 / cvb;
    const int c0 = (blockIdx.y * cvb + tx) * VN;
    if(!FIN && c0 >= C)
        return;
    const bool relu = flags & SAGA_BN_RELU;
    constexpr bool recompute = RC;
    float mean[VN], a[VN], k0[VN], k1[VN], sh[VN];
#pragma unroll
    for(int j = 0; j < VN; j++) {
        const int c = FIN && c0 >= C ? 0 : c0 + j;
        mean[j] = save_mean[c];
        sh[j] = recompute ? rb_[c] : 0.0f;
        if constexpr(!FIN) {
            a[j] = coef[c]; // s * invstd: also the forward's scale
            k0[j] = coef[C + c];
            k1[j] = coef[2 * C + c];
            sh[j] = recompute ? __builtin_fmaf(-mean[j], a[j], sh[j]) : 0.0f;
        }
    }
    typedef Ld<T, VN> L;
    typedef typename L::V V;
    // rows are walked backwards: the statistics pass that ran just before ended at the top
    const RowRun rr = row_run(rows, rb, ty, cvb_);
    const int64_t stride = rr.stride;
    const int64_t rend = rr.rend;
    auto row = [&](int64_t r) { return rows - 1 - r; };
    auto finish = [&](const V &xr, const V &gr, const V &yr, int64_t r) {
        float gv[VN], ov[VN], res[VN];
#pragma unroll
        for(int j = 0; j < VN; j++) {
            gv[j] = L::at(gr, j);
            const float yv = recompute ? (float)(T)__builtin_fmaf(L::at(xr, j), a[j], sh[j]) : L::at(yr, j);
            if(relu && !(yv > 0.0f))
                gv[j] = 0.0f;
        }
        if(beta_dx != 0.0f)
            L::load(dx + r * pdx + c0, ov);
#pragma unroll
        for(int j = 0; j < VN; j++) {
            const float v = a[j] * (gv[j] - k0[j] - (L::at(xr, j) - mean[j]) * k1[j]);
            res[j] = beta_dx != 0.0f ? v + beta_dx * ov[j] : v;
        }
        L::store(dx + r * pdx + c0, res);
        if(dz) {
            if(beta_dz != 0.0f) {
                L::load(dz + r * pdz + c0, ov);
#pragma unroll
                for(int j = 0; j < VN; j++)
                    gv[j] += beta_dz * ov[j];
            }
            L::store(dz + r * pdz + c0, gv);
        }
    };
    int64_t r = rr.r0;
    V xr[4], gr[4], yr[4];
    auto load4 = [&]() {
#pragma unroll
        for(int u = 0; u < 4; u++) {
            const int64_t q = row(r + u * stride);
            xr[u] = L::raw(x + q * px + c0);
            gr[u] = L::raw(dy + q * pdy + c0);
            yr[u] = relu && !recompute ? L::raw(y + q * py + c0) : gr[u];
        }
    };
    auto finish4 = [&]() {
#pragma unroll
        for(int u = 0; u < 4; u++)
            finish(xr[u], gr[u], yr[u], row(r + u * stride));
        r += 4 * stride;
    };
    if constexpr(FIN) {
        __shared__ float tab[3][64];
        const bool ahead = c0 < C && r + 3 * stride < rend;
        if(ahead)
            load4();
        bwd_slab(fin, C, blockIdx.y * cvb * VN, cvb * VN, tab);
        if(c0 >= C)
            return;
#pragma unroll
        for(int j = 0; j < VN; j++) {
            a[j] = tab[0][tx * VN + j];
            k0[j] = tab[1][tx * VN + j];
            k1[j] = tab[2][tx * VN + j];
            if(recompute)
                sh[j] = __builtin_fmaf(-mean[j], a[j], sh[j]);
        }
        if(ahead)
            finish4();
    }
    while(r + 3 * stride < rend) {
        load4();
        finish4();
    }
    for(; r < rend; r += stride) {
        const int64_t q = row(r);
        const V xr = L::raw(x + q * px + c0), gr = L::raw(dy + q * pdy + c0);
        finish(xr, gr, relu && !recompute ? L::raw(y + q * py + c0) : gr, q);
    }
}

// ---------------------------------------------------------------- channels-first kernels
// A channel is one plane of HW values per sample.  A block owns a contiguous run of a channel's vectors over all samples, so
// that a channel is spread over as many blocks as the tensor is worth, not one; sums leave a block as one pair, and the pass
// that follows adds a channel's pairs itself.  A thread's vectors are 256 apart; it has the loads of four on their way at once.
// us, training forward and backward with relu (one block per channel, one value at a time, which this replaces / this), fp32:
//   16 channels of 128x32x32  66 /  9, 253 / 10     64 of 128x8x8  23 /  7,  74 /  8     512 of 16x7x7  8 /  4, 12 /  4
//   16 channels of 512x32x32 534 / 16, 2370 / 39   256 of 32x56x56 175 / 53, 696 / 112   64 of 512x7x7 84 / 13, 546 / 15
// (256 of 32x56x56: forward 308 MB, backward 719 MB, 5.8 and 6.4 TB/s); two launches each are what bounds the small ones.  Channels of up to
// four vectors to a thread take one launch, in which a block holds its channel between the sums and what follows from them (us, in two launches /
// in one, forward and backward: 512 of 1x7x7 6.9 / 3.6, 7.3 / 3.7, 2048 of 8x7x7 12.2 / 6.9, 14.0 / 7.2, 64 of 1x56x56 7.0 / 4.1, 8.1 / 4.4).

constexpr int CF_HELD = 1024;      // vectors of a channel that its block holds: four to a thread
constexpr int CF_MAX_SPLITS = 256; // blocks whose sums one block adds, a pair to a thread

struct Planes {
    int64_t hwv, vectors, per; // vectors of a plane, of a channel over all samples, of a block
    int64_t HW, dn;            // values of a plane; how far 256 vectors are, in samples ...
    int dhw;                   // ... and vectors
    int splits, partials;      // blocks of a channel, and sums of it
};

// the vectors of a thread, one after the other
struct PlaneWalk {
    int64_t n, hw, i, end;
    // (held: the block has all of a channel, of CF_HELD vectors at most)
    __device__ __forceinline__ PlaneWalk(const Planes &g, int split, bool held = false)
    {
        i = held ? (int64_t)threadIdx.x : split * g.per + threadIdx.x;
        end = held || (split + 1) * g.per > g.vectors ? g.vectors : (split + 1) * g.per;
        n = held || g.vectors < 1ll << 31 ? (int64_t)((unsigned)i / (unsigned)g.hwv) : i / g.hwv;
        hw = i - n * g.hwv;
    }
    __device__ __forceinline__ void next(const Planes &g)
    {
        i += 256;
        n += g.dn;
        hw += g.dhw;
        if(hw >= g.hwv) {
            hw -= g.hwv;
            n++;
        }
    }
};

template <int N> struct PlaneBatch { // a thread's next four vectors: where they are, and whether they are
    int64_t n[N], at[N];
    bool ok[N];
    __device__ __forceinline__ void take(PlaneWalk &w, const Planes &g, int64_t c, int VN)
    {
#pragma unroll
        for(int u = 0; u < N; u++) {
            ok[u] = w.i < w.end;
            n[u] = ok[u] ? w.n : 0;
            at[u] = c * g.HW + (ok[u] ? w.hw * VN : 0);
            w.next(g);
        }
    }
};

// sums of a block's threads, for all of them
__device__ __forceinline__ void block_sum2(float &a, float &b)
{
    __shared__ float red[2][4];
    a = wave_sum(a);
    b = wave_sum(b);
    if((threadIdx.x & 63) == 0) {
        red[0][threadIdx.x >> 6] = a;
        red[1][threadIdx.x >> 6] = b;
    }
    __syncthreads();
    a = red[0][0] + red[0][1] + red[0][2] + red[0][3];
    b = red[1][0] + red[1][1] + red[1][2] + red[1][3];
}

// sums of a channel's pairs, for all threads of a block
__device__ __forceinline__ void channel_sums(const float *__restrict__ partial, int64_t c, int count, double &s0, double &s1)
{
    typedef float float2_t __attribute__((ext_vector_type(2)));
    __shared__ double red[2][4];
    const int tid = threadIdx.x;
    const float2_t v = tid < count ? ((const float2_t *)partial)[c * count + tid] : float2_t{0, 0};
    const double a0 = wave_sum_f64(v[0]), a1 = wave_sum_f64(v[1]);
    if((tid & 63) == 0) {
        red[0][tid >> 6] = a0;
        red[1][tid >> 6] = a1;
    }
    __syncthreads();
    s0 = red[0][0] + red[0][1] + red[0][2] + red[0][3];
    s1 = red[1][0] + red[1][1] + red[1][2] + red[1][3];
}

// Pass 1 of training forward: sums of (x-K) and (x-K)^2, K the channel's first value (kept: the second pass may write over it).
template <typename T, int VN>
__global__ void __launch_bounds__(256)
    bn_stats_cf(const T *__restrict__ x, int64_t npx, float *__restrict__ partial, float *__restrict__ first, Planes g)
{
    typedef Ld<T, VN, false> L;
    const int64_t c = blockIdx.x / g.splits;
    const int split = blockIdx.x - (int)c * g.splits;
    const float k = (float)x[c * g.HW];
    float a0 = 0, a1 = 0;
    PlaneWalk w(g, split);
    while(w.i < w.end) {
        PlaneBatch<4> p;
        p.take(w, g, c, VN);
        typename L::V xr[4];
#pragma unroll
        for(int u = 0; u < 4; u++)
            xr[u] = L::raw(x + p.n[u] * npx + p.at[u]);
#pragma unroll
        for(int u = 0; u < 4; u++)
            if(p.ok[u])
#pragma unroll
                for(int j = 0; j < VN; j++) {
                    const float d = L::at(xr[u], j) - k;
                    a0 += d;
                    a1 += d * d;
                }
    }
    block_sum2(a0, a1);
    if(threadIdx.x == 0) {
        partial[2 * (int64_t)blockIdx.x] = a0;
        partial[2 * (int64_t)blockIdx.x + 1] = a1;
        if(split == 0)
            first[c] = k;
    }
}

// y = x*scale[c] + shift[c] (+ z) (relu).  FROM_PAIRS: from the sums that bn_stats_cf left; FROM_HELD: from the block's own; the first block of
// a channel writes what outlives the launch.  FROM_RUNNING: run_m and run_v are the mean and the variance to normalise with.
enum { FROM_RUNNING, FROM_PAIRS, FROM_HELD };
template <typename T, int VN, int FROM>
__global__ void __launch_bounds__(256)
    bn_apply_cf(const T *x, int64_t npx, const T *z, int64_t npz, T *y, int64_t npy, const float *__restrict__ partial,
                const float *__restrict__ kept, const float *__restrict__ s, const float *__restrict__ b, float *run_m, float *run_v, float *save_mean, float *save_invstd, double M, float eps, float expavg, int flags, Planes g)
{
    typedef Ld<T, VN, false> L;
    const int64_t c = FROM == FROM_HELD ? blockIdx.x : blockIdx.x / g.splits;
    const int split = FROM == FROM_HELD ? 0 : blockIdx.x - (int)c * g.splits;
    const bool relu = flags & SAGA_BN_RELU, add = flags & SAGA_BN_ADD, first = split == 0 && threadIdx.x == 0;
    PlaneWalk w(g, split, FROM == FROM_HELD);
    PlaneBatch<4> p;
    typename L::V xr[4], zr[4];
    auto load = [&]() {
        p.take(w, g, c, VN);
#pragma unroll
        for(int u = 0; u < 4; u++) {
            xr[u] = L::raw(x + p.n[u] * npx + p.at[u]);
            zr[u] = add ? L::raw(z + p.n[u] * npz + p.at[u]) : xr[u];
        }
    };
    // (a thread without a vector requests the channel's first: all have to meet below)
    bool more = w.i < w.end;
    load();
    float sc, sh;
    if constexpr(FROM != FROM_RUNNING) {
        // (y may be x: nobody writes before the sums have met)
        const float k = FROM == FROM_HELD ? (float)x[c * g.HW] : kept[c], sv = s[c], bv = b[c];
        const float rm = first && run_m ? run_m[c] : 0.0f, rv = first && run_v ? run_v[c] : 0.0f;
        double s0, s1;
        if constexpr(FROM == FROM_HELD) {
            float a0 = 0, a1 = 0;
#pragma unroll
            for(int u = 0; u < 4; u++)
                if(p.ok[u])
#pragma unroll
                    for(int j = 0; j < VN; j++) {
                        const float d = L::at(xr[u], j) - k;
                        a0 += d;
                        a1 += d * d;
                    }
            block_sum2(a0, a1);
            s0 = a0;
            s1 = a1;
        } else {
            channel_sums(partial, c, g.partials, s0, s1);
        }
        finish_stats(s0, s1, k, M, eps, expavg, sv, bv, rm, rv, first, run_m, run_v, save_mean, save_invstd, (int)c, sc, sh);
    } else {
        sc = s[c] * rsqrtf(run_v[c] + eps);
        sh = b[c] - run_m[c] * sc;
    }
    while(more) {
#pragma unroll
        for(int u = 0; u < 4; u++) {
            if(!p.ok[u])
                continue;
            float o[VN];
#pragma unroll
            for(int j = 0; j < VN; j++) {
                float t = __builtin_fmaf(L::at(xr[u], j), sc, sh);
                if(add)
                    t += L::at(zr[u], j);
                if(relu)
                    t = (t != t) ? t : fmaxf(t, 0.0f);
                o[j] = t;
            }
            L::store(y + p.n[u] * npy + p.at[u], o);
        }
        more = FROM != FROM_HELD && w.i < w.end;
        if(more)
            load();
    }
}

// Inference, vectors in the order of memory, whatever their channel is (infer_in_order).
template <typename T, int VN>
__global__ void __launch_bounds__(256)
    bn_infer_cf(const T *x, int64_t npx, const T *z, int64_t npz, T *y, int64_t npy, const float *__restrict__ s, const float *__restrict__ b,
                const float *__restrict__ m, const float *__restrict__ v, float eps, int flags, int C, unsigned hwv, unsigned total)
{
    typedef Ld<T, VN, false> L;
    const bool relu = flags & SAGA_BN_RELU, add = flags & SAGA_BN_ADD;
    for(unsigned i = blockIdx.x * 256 + threadIdx.x; i < total; i += gridDim.x * 256) {
        const unsigned nc = i / hwv, n = nc / (unsigned)C, c = nc - n * (unsigned)C;
        const int64_t at = ((int64_t)c * hwv + (i - nc * hwv)) * VN;
        const auto xr = L::raw(x + n * npx + at);
        const auto zr = add ? L::raw(z + n * npz + at) : xr;
        const float sc = s[c] * rsqrtf(v[c] + eps), sh = b[c] - m[c] * sc;
        float o[VN];
#pragma unroll
        for(int j = 0; j < VN; j++) {
            float t = __builtin_fmaf(L::at(xr, j), sc, sh);
            if(add)
                t += L::at(zr, j);
            if(relu)
                t = (t != t) ? t : fmaxf(t, 0.0f);
            o[j] = t;
        }
        L::store(y + n * npy + at, o);
    }
}

// Pass 1 of backward: sums of dy' and dy'*(x-mean); dy' = dy, zero where the relu's y is.  dz set: dy' goes there on the way,
// and the second pass reads it in place of y and dy.
template <typename T, int VN>
__global__ void __launch_bounds__(256)
    bn_bwd_stats_cf(const T *__restrict__ x, int64_t npx, const T *__restrict__ y, int64_t npy, const T *__restrict__ dy, int64_t npdy,
                    T *__restrict__ dz, int64_t npdz, const float *__restrict__ save_mean, float *__restrict__ partial, Planes g)
{
    typedef Ld<T, VN, false> L;
    const int64_t c = blockIdx.x / g.splits;
    const int split = blockIdx.x - (int)c * g.splits;
    const float mean = save_mean[c];
    float a0 = 0, a1 = 0;
    PlaneWalk w(g, split);
    while(w.i < w.end) {
        PlaneBatch<4> p;
        p.take(w, g, c, VN);
        typename L::V xr[4], gr[4], yr[4];
#pragma unroll
        for(int u = 0; u < 4; u++) {
            xr[u] = L::raw(x + p.n[u] * npx + p.at[u]);
            gr[u] = L::raw(dy + p.n[u] * npdy + p.at[u]);
            yr[u] = y ? L::raw(y + p.n[u] * npy + p.at[u]) : gr[u];
        }
#pragma unroll
        for(int u = 0; u < 4; u++) {
            if(!p.ok[u])
                continue;
            float gm[VN];
#pragma unroll
            for(int j = 0; j < VN; j++) {
                gm[j] = y && !(L::at(yr[u], j) > 0.0f) ? 0.0f : L::at(gr[u], j);
                a0 += gm[j];
                a1 += gm[j] * (L::at(xr[u], j) - mean);
            }
            if(dz)
                L::store(dz + p.n[u] * npdz + p.at[u], gm);
        }
    }
    block_sum2(a0, a1);
    if(threadIdx.x == 0) {
        partial[2 * (int64_t)blockIdx.x] = a0;
        partial[2 * (int64_t)blockIdx.x + 1] = a1;
    }
}

// Pass 2 of backward: dx = s*invstd*(dy' - db/M - (x-mean)*invstd*ds/M) ; dz = dy'.  HELD: and pass 1, of what the block holds.
template <typename T, int VN, bool HELD>
__global__ void __launch_bounds__(256)
    bn_bwd_apply_cf(const T *x, int64_t npx, const T *y, int64_t npy, const T *dy, int64_t npdy, T *dx, int64_t npdx, T *dz,
                    int64_t npdz, const float *__restrict__ partial, const float *__restrict__ s,
                    const float *__restrict__ save_mean, const float *__restrict__ save_invstd, float *ds, float *db, double M,
                    float beta_dx, float beta_dz, float beta_p, Planes g)
{
    typedef Ld<T, VN, false> L;
    const int64_t c = HELD ? blockIdx.x : blockIdx.x / g.splits;
    const int split = HELD ? 0 : blockIdx.x - (int)c * g.splits;
    const bool first = split == 0 && threadIdx.x == 0;
    PlaneWalk w(g, split, HELD);
    PlaneBatch<4> p;
    typename L::V xr[4], gr[4], yr[4];
    auto load = [&]() {
        p.take(w, g, c, VN);
#pragma unroll
        for(int u = 0; u < 4; u++) {
            xr[u] = L::raw(x + p.n[u] * npx + p.at[u]);
            gr[u] = L::raw(dy + p.n[u] * npdy + p.at[u]);
            yr[u] = y ? L::raw(y + p.n[u] * npy + p.at[u]) : gr[u];
        }
    };
    bool more = w.i < w.end;
    load();
    const float mean = save_mean[c], inv = save_invstd[c], sv = s[c];
    const float ds_old = first && beta_p != 0.0f ? ds[c] : 0.0f, db_old = first && beta_p != 0.0f ? db[c] : 0.0f;
    double s0, s1;
    if constexpr(HELD) { // (dx and dz may be what was read: nobody writes before the sums have met)
        float a0 = 0, a1 = 0;
#pragma unroll
        for(int u = 0; u < 4; u++)
            if(p.ok[u])
#pragma unroll
                for(int j = 0; j < VN; j++) {
                    const float gm = y && !(L::at(yr[u], j) > 0.0f) ? 0.0f : L::at(gr[u], j);
                    a0 += gm;
                    a1 += gm * (L::at(xr[u], j) - mean);
                }
        block_sum2(a0, a1);
        s0 = a0;
        s1 = a1;
    } else {
        channel_sums(partial, c, g.partials, s0, s1);
    }
    const double dsv = s1 * inv;
    if(first) {
        ds[c] = (float)(beta_p != 0.0f ? dsv + (double)beta_p * ds_old : dsv);
        db[c] = (float)(beta_p != 0.0f ? s0 + (double)beta_p * db_old : s0);
    }
    const float a = (float)(sv * (double)inv), k0 = (float)(s0 / M), k1 = (float)(dsv * inv / M);
    while(more) {
#pragma unroll
        for(int u = 0; u < 4; u++) {
            if(!p.ok[u])
                continue;
            float gv[VN], ov[VN], res[VN];
            T *const pd = dx + p.n[u] * npdx + p.at[u];
            if(beta_dx != 0.0f)
                L::load(pd, ov);
#pragma unroll
            for(int j = 0; j < VN; j++) {
                gv[j] = y && !(L::at(yr[u], j) > 0.0f) ? 0.0f : L::at(gr[u], j);
                const float v = a * (gv[j] - k0 - (L::at(xr[u], j) - mean) * k1);
                res[j] = beta_dx != 0.0f ? v + beta_dx * ov[j] : v;
            }
            L::store(pd, res);
            if(dz) {
                T *const pz = dz + p.n[u] * npdz + p.at[u];
                if(beta_dz != 0.0f) {
                    L::load(pz, ov);
#pragma unroll
                    for(int j = 0; j < VN; j++)
                        gv[j] += beta_dz * ov[j];
                }
                L::store(pz, gv);
            }
        }
        more = !HELD && w.i < w.end;
        if(more)
            load();
    }
}

// ---------------------------------------------------------------- host side

struct Views {
    bool cl;
    CLInfo lx, ly, lz, ldy, ldx, ldz;
    CFInfo fx, fy, fz, fdy, fdx, fdz;
};

static int vec_width(int dtype, int C, std::initializer_list<const SagaTensorView *> vs,
                     std::initializer_list<int64_t> pitches)
{
    const int vn = dtype == SAGA_HALF ? 8 : 4;
    if(C % vn)
        return 1;
    for(auto v : vs)
        if(v && !aligned16(v->ptr))
            return 1;
    for(auto p : pitches)
        if(p % vn)
            return 1;
    return vn;
}

// the same for planes
static int cf_vec_width(int dtype, const CFInfo &f, std::initializer_list<std::pair<const SagaTensorView *, int64_t>> vs)
{
    const int vn = dtype == SAGA_HALF ? 8 : 4;
    if(f.HW % vn)
        return 1;
    for(const auto &v : vs)
        if(v.first && (!aligned16(v.first->ptr) || v.second % vn))
            return 1;
    return vn;
}

// SAGA_HIP_BN_GRIDSTRIDE: bits select the kernels that walk their rows grid-strided (row_run)
// (1 forward apply, 2 forward statistics, 4 backward statistics, 8 backward apply); default: the two apply passes
static int gridstride_mask()
{
    static const int v = env_int("SAGA_HIP_BN_GRIDSTRIDE", 9);
    return v;
}
#define WALK_CVB(bit) ((gridstride_mask() & (bit)) ? -sh.cvb : sh.cvb)
#define WALK_GRID(bit) ((gridstride_mask() & (bit)) ? dim3(sh.gx, sh.gy) : dim3(sh.gxa, sh.gy))

static bool force_y_mask()
{
    static int v = -1;
    if(v < 0) {
        const char *e = getenv("SAGA_HIP_BN_MASK_FROM_Y");
        v = (e && *e && *e != '0') ? 1 : 0;
    }
    return v == 1;
}

// Vectors of a plane of several samples, and blocks with about four of them per thread (at most some 8192, and at most `most` of a channel).
static Planes plan_planes(const CFInfo &f, int vn, int64_t most)
{
    Planes g;
    g.HW = f.HW;
    g.hwv = f.HW / vn;
    g.vectors = g.hwv * f.N;
    g.dn = 256 / g.hwv;
    g.dhw = (int)(256 - g.dn * g.hwv);
    int64_t splits = std::min((g.vectors + 1023) / 1024, std::min(most, std::max<int64_t>(1, 8192 / f.C)));
    g.per = ((g.vectors + splits - 1) / splits + 255) / 256 * 256;
    g.splits = g.partials = (int)((g.vectors + g.per - 1) / g.per);
    return g;
}

// Whether inference takes the vectors in the order of memory (bn_infer_cf).  In the order of the channels neighbouring lanes are planes apart
// where planes are small, and a block waits for its channel's numbers before it has four vectors' work to do.  us, by channel / in order:
// fp32 512x64x2x2 4.4 / 2.5, 512x512x3x3 13.1 / 7.9, 1x64x56x56 3.5 / 2.5, 64x256x14x14 6.6 / 5.2, 1024x512x4x4 17.7 / 12.4, 64x1024x13x13 24 / 24.  Single
// values of two bytes are the exception once there are many: 512x512x7x7 23 / 27, 2x16x300x301 7.2 / 8.1, 64x256x14x14 8.2 / 8.9; 512x512x6x6 22 / 20.
static bool infer_in_order(const Planes &g, int C, int vn, int dtype)
{
    const int64_t total = g.vectors * C;
    return total < 1ll << 31 && !(vn == 1 && dtype == SAGA_HALF && g.HW >= 49 && total >= 1 << 21);
}

// The blocks of a channel whose sums the workspace has room for: it is sized by the plans for channels-last tensors.
static int64_t cf_room(const CFInfo &f) { return std::min<int64_t>(CF_MAX_SPLITS, plan((int64_t)f.N * f.HW, f.C).gx); }

static size_t ws_floats(int64_t rows, int C, int dtype)
{
    // partials for the widest plan (vector width 1 gives the most blocks along y) + 3*C coefficients
    size_t best = 0;
    for(int vn : {1, dtype == SAGA_HALF ? 8 : 4}) {
        if(C % vn)
            continue;
        Shape sh = plan(rows, C / vn);
        size_t need = (size_t)sh.gx * C * 2;
        if(need > best)
            best = need;
    }
    return best + 3 * (size_t)C + 64;
}

} // namespace

int bn_launch_bwd_finalize(const float *partial, int rows, const float *s, const float *save_invstd, float *ds, float *db,
                           float *coef, double M, int C, float beta_p, hipStream_t st)
{
    bn_bwd_finalize<<<C, 256, 0, st>>>(partial, rows, s, save_invstd, ds, db, coef, M, C, beta_p);
    SAGA_CHECK_LAUNCH();
    return 0;
}

extern "C" {

size_t saga_hip_bn_workspace_size(const SagaTensorView *x)
{
    if(!x)
        return 0;
    const int64_t rows = (int64_t)x->dims[0] * x->dims[2] * x->dims[3];
    return ws_floats(rows, x->dims[1], x->dtype) * sizeof(float);
}

int saga_hip_bn_infer(const SagaTensorView *x, const SagaTensorView *z, const SagaTensorView *y, const float *s,
                      const float *b, const float *m, const float *v, float eps, int flags, saga_stream_t stream)
{
    if(!valid_view(x) || !valid_view(y) || !s || !b || !m || !v)
        return SAGA_HIP_EINVAL;
    const bool add = flags & SAGA_BN_ADD;
    if(add && !valid_view(z))
        return SAGA_HIP_EINVAL;
    if(!same_dims(x, y) || (add && !same_dims(x, z)))
        return SAGA_HIP_ESHAPE;
    if(x->dtype != y->dtype || (add && z->dtype != x->dtype) || (x->dtype != SAGA_HALF && x->dtype != SAGA_FLOAT))
        return SAGA_HIP_EUNSUPPORTED;
    hipStream_t st = as_stream(stream);
    CLInfo lx, ly, lz = {};
    CFInfo fx, fy, fz = {};
    if(as_channels_last(x, &lx) && as_channels_last(y, &ly) && (!add || as_channels_last(z, &lz))) {
        const int vn = vec_width(x->dtype, lx.C, {x, y, add ? z : nullptr}, {lx.pitch, ly.pitch, add ? lz.pitch : 0});
        Shape sh = plan(lx.rows, lx.C / vn);
        dim3 grid(sh.gx, sh.gy);
#define GO(T, VN)                                                                                                 \
    bn_apply_cl<T, VN, 0><<<WALK_GRID(1), 256, 0, st>>>((const T *)x->ptr, lx.pitch, add ? (const T *)z->ptr : nullptr,      \
                                                lz.pitch, (T *)y->ptr, ly.pitch, s, b, m, v, nullptr, eps, lx.rows, \
                                                lx.C, WALK_CVB(1), flags)
        if(x->dtype == SAGA_HALF) {
            if(vn == 8) GO(half_t, 8); else GO(half_t, 1);
        } else {
            if(vn == 4) GO(float, 4); else GO(float, 1);
        }
#undef GO
    } else if(as_channels_first(x, &fx) && as_channels_first(y, &fy) && (!add || as_channels_first(z, &fz))) {
        const int vn = cf_vec_width(x->dtype, fx, {{x, fx.npitch}, {y, fy.npitch}, {add ? z : nullptr, fz.npitch}});
        const Planes g = plan_planes(fx, vn, 1 << 16);
        const int64_t total = g.vectors * fx.C;
        if(infer_in_order(g, fx.C, vn, x->dtype)) {
#define GO(T, VN)                                                                                                                 \
    bn_infer_cf<T, VN><<<grid_for(total, 256, 256 * 32), 256, 0, st>>>((const T *)x->ptr, fx.npitch, add ? (const T *)z->ptr : nullptr, fz.npitch, \
                                                                       (T *)y->ptr, fy.npitch, s, b, m, v, eps, flags, fx.C, (unsigned)g.hwv,      \
                                                                       (unsigned)total)
            if(x->dtype == SAGA_HALF) {
                if(vn == 8) GO(half_t, 8); else GO(half_t, 1);
            } else {
                if(vn == 4) GO(float, 4); else GO(float, 1);
            }
#undef GO
            SAGA_CHECK_LAUNCH();
            return 0;
        }
#define GO(T, VN)                                                                                                                 \
    bn_apply_cf<T, VN, FROM_RUNNING><<<(unsigned)(g.splits * (int64_t)fx.C), 256, 0, st>>>(                                              \
        (const T *)x->ptr, fx.npitch, add ? (const T *)z->ptr : nullptr, fz.npitch, (T *)y->ptr, fy.npitch, nullptr, nullptr, s, b, \
        (float *)m, (float *)v, nullptr, nullptr, 0.0, eps, 0.0f, flags, g)
        if(x->dtype == SAGA_HALF) {
            if(vn == 8) GO(half_t, 8); else GO(half_t, 1);
        } else {
            if(vn == 4) GO(float, 4); else GO(float, 1);
        }
#undef GO
    } else {
        return SAGA_HIP_EUNSUPPORTED;
    }
    SAGA_CHECK_LAUNCH();
    return 0;
}

int saga_hip_bn_train_fwd(const SagaTensorView *x, const SagaTensorView *z, const SagaTensorView *y,
                          const float *s, const float *b, float *run_m, float *run_v, float *save_mean,
                          float *save_invstd, float eps, float expavg, int flags, void *workspace,
                          size_t ws_bytes, saga_stream_t stream)
{
    if(!valid_view(x) || !valid_view(y) || !s || !b)
        return SAGA_HIP_EINVAL;
    const bool add = flags & SAGA_BN_ADD;
    if(add && !valid_view(z))
        return SAGA_HIP_EINVAL;
    if(!same_dims(x, y) || (add && !same_dims(x, z)))
        return SAGA_HIP_ESHAPE;
    if(x->dtype != y->dtype || (add && z->dtype != x->dtype) || (x->dtype != SAGA_HALF && x->dtype != SAGA_FLOAT))
        return SAGA_HIP_EUNSUPPORTED;
    if(!workspace || ws_bytes < saga_hip_bn_workspace_size(x))
        return SAGA_HIP_EWORKSPACE;
    hipStream_t st = as_stream(stream);
    float *ws = (float *)workspace;
    CLInfo lx, ly, lz = {};
    CFInfo fx, fy, fz = {};
    if(as_channels_last(x, &lx) && as_channels_last(y, &ly) && (!add || as_channels_last(z, &lz))) {
        const int C = lx.C;
        const int vn = vec_width(x->dtype, C, {x, y, add ? z : nullptr}, {lx.pitch, ly.pitch, add ? lz.pitch : 0});
        Shape sh = plan(lx.rows, C / vn);
        dim3 grid(sh.gx, sh.gy);
        float *partial = ws, *ss = ws + (size_t)sh.gx * C * 2;
#define GO(T, VN)                                                                                                   \
    do {                                                                                                            \
        bn_stats_cl<T, VN><<<grid, 256, 0, st>>>((const T *)x->ptr, lx.pitch, partial, lx.rows, C, WALK_CVB(2));           \
        bn_stats_finalize<T><<<C, 256, 0, st>>>(partial, sh.gx, (const T *)x->ptr, 1, s, b, run_m,      \
                                                              run_v, save_mean, save_invstd, ss, (double)lx.rows, C, \
                                                              eps, expavg);                                         \
        bn_apply_cl<T, VN, 1><<<WALK_GRID(1), 256, 0, st>>>((const T *)x->ptr, lx.pitch, add ? (const T *)z->ptr : nullptr,   \
                                                    lz.pitch, (T *)y->ptr, ly.pitch, nullptr, nullptr, nullptr,     \
                                                    nullptr, ss, eps, lx.rows, C, WALK_CVB(1), flags);                   \
    } while(0)
        if(x->dtype == SAGA_HALF) {
            if(vn == 8) GO(half_t, 8); else GO(half_t, 1);
        } else {
            if(vn == 4) GO(float, 4); else GO(float, 1);
        }
#undef GO
    } else if(as_channels_first(x, &fx) && as_channels_first(y, &fy) && (!add || as_channels_first(z, &fz))) {
        const int vn = cf_vec_width(x->dtype, fx, {{x, fx.npitch}, {y, fy.npitch}, {add ? z : nullptr, fz.npitch}});
        const Planes g1 = plan_planes(fx, vn, cf_room(fx));
        Planes g2 = plan_planes(fx, vn, 1 << 16);
        g2.partials = g1.partials;
        float *const kept = ws + 2 * (int64_t)fx.C * g1.splits;
        const double M = (double)fx.N * fx.HW;
        const bool held = g2.vectors <= CF_HELD;
#define GO(T, VN)                                                                                                                 \
    do {                                                                                                                          \
        if(!held)                                                                                                                 \
            bn_stats_cf<T, VN><<<(unsigned)(g1.splits * (int64_t)fx.C), 256, 0, st>>>((const T *)x->ptr, fx.npitch, ws, kept, g1); \
        auto kern = held ? bn_apply_cf<T, VN, FROM_HELD> : bn_apply_cf<T, VN, FROM_PAIRS>;                                        \
        kern<<<(unsigned)(g2.splits * (int64_t)fx.C), 256, 0, st>>>(                                                              \
            (const T *)x->ptr, fx.npitch, add ? (const T *)z->ptr : nullptr, fz.npitch, (T *)y->ptr, fy.npitch, ws, kept, s, b,   \
            run_m, run_v, save_mean, save_invstd, M, eps, expavg, flags, g2);                                                     \
    } while(0)
        if(x->dtype == SAGA_HALF) {
            if(vn == 8) GO(half_t, 8); else GO(half_t, 1);
        } else {
            if(vn == 4) GO(float, 4); else GO(float, 1);
        }
#undef GO
    } else {
        return SAGA_HIP_EUNSUPPORTED;
    }
    SAGA_CHECK_LAUNCH();
    return 0;
}

int saga_hip_bn_train_fwd_partials(const SagaTensorView *x, const SagaTensorView *z, const SagaTensorView *y,
                                   const float *s, const float *b, float *run_m, float *run_v, float *save_mean,
                                   float *save_invstd, float eps, float expavg, int flags, const float *partial,
                                   int partial_rows, uint8_t *relu_mask, void *workspace, size_t ws_bytes,
                                   saga_stream_t stream)
{
    if(!valid_view(x) || (y && !valid_view(y)) || !s || !b || !partial || partial_rows < 1)
        return SAGA_HIP_EINVAL;
    if(!y) {
        // statistics only: mean, 1/std and the running statistics as usual, and scale[c], shift[c] (2*C floats)
        // into the workspace, for a consumer that applies them itself (saga_hip_maxpool_fwd_codes_bn)
        if(z || relu_mask || (x->dtype != SAGA_HALF && x->dtype != SAGA_FLOAT))
            return SAGA_HIP_EINVAL;
        const int C = x->dims[1];
        if(!workspace || ws_bytes < 2 * (size_t)C * sizeof(float))
            return SAGA_HIP_EWORKSPACE;
        const double rows = (double)x->dims[0] * x->dims[2] * x->dims[3];
        if(x->dtype == SAGA_HALF)
            bn_stats_finalize<half_t><<<C, 256, 0, as_stream(stream)>>>(partial, partial_rows, (const half_t *)nullptr, 1, s, b,
                                                                        run_m, run_v, save_mean, save_invstd,
                                                                        (float *)workspace, rows, C, eps, expavg);
        else
            bn_stats_finalize<float><<<C, 256, 0, as_stream(stream)>>>(partial, partial_rows, (const float *)nullptr, 1, s, b,
                                                                       run_m, run_v, save_mean, save_invstd,
                                                                       (float *)workspace, rows, C, eps, expavg);
        SAGA_CHECK_LAUNCH();
        return 0;
    }
    const bool add = flags & SAGA_BN_ADD;
    if(add && !valid_view(z))
        return SAGA_HIP_EINVAL;
    if(!same_dims(x, y) || (add && !same_dims(x, z)))
        return SAGA_HIP_ESHAPE;
    if(x->dtype != y->dtype || (add && z->dtype != x->dtype) || (x->dtype != SAGA_HALF && x->dtype != SAGA_FLOAT))
        return SAGA_HIP_EUNSUPPORTED;
    CLInfo lx, ly, lz = {};
    if(!as_channels_last(x, &lx) || !as_channels_last(y, &ly) || (add && !as_channels_last(z, &lz)))
        return SAGA_HIP_EUNSUPPORTED;
    const int C = lx.C;
    if(!workspace || ws_bytes < 2 * (size_t)C * sizeof(float))
        return SAGA_HIP_EWORKSPACE;
    hipStream_t st = as_stream(stream);
    float *ss = (float *)workspace;
    const int vn = vec_width(x->dtype, C, {x, y, add ? z : nullptr}, {lx.pitch, ly.pitch, add ? lz.pitch : 0});
    // the mask has one byte per 8 fp16 channels: only the 8-wide fp16 kernel with relu writes it
    if(relu_mask && !(x->dtype == SAGA_HALF && vn == 8 && (flags & SAGA_BN_RELU)))
        return SAGA_HIP_EUNSUPPORTED;
    Shape sh;
    if(x->dtype == SAGA_HALF && vn == 8 && self_finalizing(lx.rows, C, partial_rows, false, &sh)) {
        const StatsFin fin = {partial, partial_rows, s, b, run_m, run_v, save_mean, save_invstd, (double)lx.rows, eps, expavg};
        bn_apply_cl<half_t, 8, 2><<<dim3(sh.gx, sh.gy), 256, 0, st>>>(
            (const half_t *)x->ptr, lx.pitch, add ? (const half_t *)z->ptr : nullptr, lz.pitch, (half_t *)y->ptr, ly.pitch, nullptr,
            nullptr, nullptr, nullptr, nullptr, eps, lx.rows, C, sh.cvb, flags, relu_mask, fin);
        SAGA_CHECK_LAUNCH();
        return 0;
    }
    sh = plan(lx.rows, C / vn);
#define GO(T, VN)                                                                                                   \
    do {                                                                                                            \
        bn_stats_finalize<T><<<C, 256, 0, st>>>(partial, partial_rows, (const T *)nullptr, 1, s, b, run_m, \
                                                          run_v, save_mean, save_invstd, ss, (double)lx.rows, C,    \
                                                          eps, expavg);                                             \
        bn_apply_cl<T, VN, 1><<<WALK_GRID(1), 256, 0, st>>>((const T *)x->ptr, lx.pitch, add ? (const T *)z->ptr : nullptr,   \
                                                    lz.pitch, (T *)y->ptr, ly.pitch, nullptr, nullptr, nullptr,     \
                                                    nullptr, ss, eps, lx.rows, C, WALK_CVB(1), flags, relu_mask);        \
    } while(0)
    if(x->dtype == SAGA_HALF) {
        if(vn == 8) GO(half_t, 8); else GO(half_t, 1);
    } else {
        if(vn == 4) GO(float, 4); else GO(float, 1);
    }
#undef GO
    SAGA_CHECK_LAUNCH();
    return 0;
}

int saga_hip_bn_bwd(const SagaTensorView *x, const SagaTensorView *y, const SagaTensorView *dy,
                    const SagaTensorView *dx, const SagaTensorView *dz, const float *s, const float *save_mean,
                    const float *save_invstd, float *ds, float *db, float beta_dx, float beta_dz, float beta_p,
                    int flags, void *workspace, size_t ws_bytes, saga_stream_t stream)
{
    return saga_hip_bn_bwd_ex(x, y, dy, dx, dz, s, nullptr, save_mean, save_invstd, ds, db, beta_dx, beta_dz, beta_p,
                              flags, nullptr, workspace, ws_bytes, stream);
}

int saga_hip_bn_bwd_ex(const SagaTensorView *x, const SagaTensorView *y, const SagaTensorView *dy,
                       const SagaTensorView *dx, const SagaTensorView *dz, const float *s, const float *b,
                       const float *save_mean, const float *save_invstd, float *ds, float *db, float beta_dx,
                       float beta_dz, float beta_p, int flags, const uint8_t *relu_mask, void *workspace,
                       size_t ws_bytes, saga_stream_t stream)
{
    if(!valid_view(x) || !valid_view(dy) || !valid_view(dx) || !s || !save_mean || !save_invstd || !ds || !db)
        return SAGA_HIP_EINVAL;
    bool relu = flags & SAGA_BN_RELU;
    // with the bias at hand and no residual, the relu mask is a function of x: y is not needed
    CLInfo cl_probe;
    const bool recompute = relu && b && !(flags & SAGA_BN_ADD) && !force_y_mask() && as_channels_last(x, &cl_probe) &&
                           as_channels_last(dy, &cl_probe) && as_channels_last(dx, &cl_probe);
    if(relu && !recompute && !valid_view(y))
        return SAGA_HIP_EINVAL;
    if(recompute)
        y = nullptr;
    const bool need_y = relu && !recompute;
    relu = need_y; // below, "relu" guards every use of y
    if(dz && !valid_view(dz))
        return SAGA_HIP_EINVAL;
    if(!same_dims(x, dy) || !same_dims(x, dx) || (relu && !same_dims(x, y)) || (dz && !same_dims(x, dz)))
        return SAGA_HIP_ESHAPE;
    const int dt = x->dtype;
    if((dt != SAGA_HALF && dt != SAGA_FLOAT) || dy->dtype != dt || dx->dtype != dt || (relu && y->dtype != dt) ||
       (dz && dz->dtype != dt))
        return SAGA_HIP_EUNSUPPORTED;
    if(!workspace || ws_bytes < saga_hip_bn_workspace_size(x))
        return SAGA_HIP_EWORKSPACE;
    hipStream_t st = as_stream(stream);
    float *ws = (float *)workspace;
    CLInfo lx, ly = {}, ldy, ldx, ldz = {};
    CFInfo fx, fy = {}, fdy, fdx, fdz = {};
    if(as_channels_last(x, &lx) && as_channels_last(dy, &ldy) && as_channels_last(dx, &ldx) &&
       (!relu || as_channels_last(y, &ly)) && (!dz || as_channels_last(dz, &ldz))) {
        const int C = lx.C;
        const int vn = vec_width(dt, C, {x, dy, dx, relu ? y : nullptr, dz},
                                 {lx.pitch, ldy.pitch, ldx.pitch, relu ? ly.pitch : 0, dz ? ldz.pitch : 0});
        Shape sh = plan(lx.rows, C / vn, true);
        dim3 grid(sh.gx, sh.gy);
        float *partial = ws, *coef = ws + (size_t)sh.gx * C * 2;
        // residual layers: the first pass leaves dy' in dz, the second reads it in place of y and dy
        const bool early_dz = dz && beta_dz == 0.0f && relu && !recompute && dz->ptr != dy->ptr && dz->ptr != x->ptr &&
                              dz->ptr != y->ptr;
        // the forward pass's relu mask replaces y where only the first pass needs it
        const uint8_t *mk = relu_mask && early_dz && dt == SAGA_HALF && vn == 8 ? relu_mask : nullptr;
#define GO(T, VN)                                                                                                    \
    do {                                                                                                             \
        if(recompute)                                                                                                \
            GO2(T, VN, true);                                                                                        \
        else                                                                                                         \
            GO2(T, VN, false);                                                                                       \
    } while(0)
#define GO2(T, VN, RC)                                                                                               \
    do {                                                                                                             \
        bn_bwd_stats_cl<T, VN, RC><<<grid, 256, 0, st>>>((const T *)x->ptr, lx.pitch, relu ? (const T *)y->ptr : nullptr,  \
                                                     ly.pitch, (const T *)dy->ptr, ldy.pitch, save_mean, partial,    \
                                                     lx.rows, C, WALK_CVB(4), flags, recompute ? s : nullptr,             \
                                                     recompute ? b : nullptr, recompute ? save_invstd : nullptr,     \
                                                     early_dz ? (T *)dz->ptr : nullptr, ldz.pitch, mk);              \
        if constexpr(sizeof(T) == 2 && VN == 8) {                                                                    \
            Shape sf;                                                                                                \
            if(self_finalizing(lx.rows, C, sh.gx, true, &sf)) {                                                            \
                const BwdFin fin = {partial, sh.gx, s, save_invstd, ds, db, (double)lx.rows, beta_p};                \
                if(early_dz)                                                                                         \
                    bn_bwd_apply_cl<T, VN, false, true><<<dim3(sf.gx, sf.gy), 256, 0, st>>>(                         \
                        (const T *)x->ptr, lx.pitch, nullptr, 0, (const T *)dz->ptr, ldz.pitch, (T *)dx->ptr,        \
                        ldx.pitch, nullptr, 0, save_mean, coef, lx.rows, C, sf.cvb, flags & ~SAGA_BN_RELU, beta_dx,  \
                        0.0f, nullptr, fin);                                                                         \
                else                                                                                                 \
                    bn_bwd_apply_cl<T, VN, RC, true><<<dim3(sf.gx, sf.gy), 256, 0, st>>>(                            \
                        (const T *)x->ptr, lx.pitch, relu ? (const T *)y->ptr : nullptr, ly.pitch,                   \
                        (const T *)dy->ptr, ldy.pitch, (T *)dx->ptr, ldx.pitch, dz ? (T *)dz->ptr : nullptr,         \
                        ldz.pitch, save_mean, coef, lx.rows, C, sf.cvb, flags, beta_dx, beta_dz,                     \
                        recompute ? b : nullptr, fin);                                                               \
                break;                                                                                               \
            }                                                                                                        \
        }                                                                                                            \
        bn_bwd_finalize<<<C, 256, 0, st>>>(partial, sh.gx, s, save_invstd, ds, db, coef,                \
                                                         (double)lx.rows, C, beta_p);                                \
        if(early_dz)                                                                                                 \
            bn_bwd_apply_cl<T, VN, false><<<WALK_GRID(8), 256, 0, st>>>((const T *)x->ptr, lx.pitch, nullptr, 0,              \
                                                                (const T *)dz->ptr, ldz.pitch, (T *)dx->ptr,          \
                                                                ldx.pitch, nullptr, 0, save_mean, coef, lx.rows, C,   \
                                                                WALK_CVB(8), flags & ~SAGA_BN_RELU, beta_dx, 0.0f,         \
                                                                nullptr);                                             \
        else                                                                                                         \
            bn_bwd_apply_cl<T, VN, RC><<<WALK_GRID(8), 256, 0, st>>>(                                                        \
                (const T *)x->ptr, lx.pitch, relu ? (const T *)y->ptr : nullptr, ly.pitch, (const T *)dy->ptr,       \
                ldy.pitch, (T *)dx->ptr, ldx.pitch, dz ? (T *)dz->ptr : nullptr, ldz.pitch, save_mean, coef,         \
                lx.rows, C, WALK_CVB(8), flags, beta_dx, beta_dz, recompute ? b : nullptr);                               \
    } while(0)
        if(dt == SAGA_HALF) {
            if(vn == 8) GO(half_t, 8); else GO(half_t, 1);
        } else {
            if(vn == 4) GO(float, 4); else GO(float, 1);
        }
#undef GO
#undef GO2
    } else if(!recompute && as_channels_first(x, &fx) && as_channels_first(dy, &fdy) && as_channels_first(dx, &fdx) &&
              (!relu || as_channels_first(y, &fy)) && (!dz || as_channels_first(dz, &fdz))) {
        const int vn = cf_vec_width(dt, fx, {{x, fx.npitch}, {dy, fdy.npitch}, {dx, fdx.npitch}, {relu ? y : nullptr, fy.npitch}, {dz, fdz.npitch}});
        const Planes g1 = plan_planes(fx, vn, cf_room(fx));
        Planes g2 = plan_planes(fx, vn, 1 << 16);
        g2.partials = g1.partials;
        const double M = (double)fx.N * fx.HW;
        const bool held = g2.vectors <= CF_HELD;
        // (as above: the first pass leaves dy' in dz)
        const bool early_dz = !held && dz && beta_dz == 0.0f && relu && dz->ptr != dy->ptr && dz->ptr != x->ptr && dz->ptr != y->ptr;
#define GO(T, VN)                                                                                                                 \
    do {                                                                                                                          \
        T *const zp = dz ? (T *)dz->ptr : nullptr;                                                                                \
        const T *const yp = relu ? (const T *)y->ptr : nullptr;                                                                   \
        if(!held)                                                                                                                 \
            bn_bwd_stats_cf<T, VN><<<(unsigned)(g1.splits * (int64_t)fx.C), 256, 0, st>>>(                                        \
                (const T *)x->ptr, fx.npitch, yp, fy.npitch, (const T *)dy->ptr, fdy.npitch, early_dz ? zp : nullptr, fdz.npitch, \
                save_mean, ws, g1);                                                                                               \
        auto kern = held ? bn_bwd_apply_cf<T, VN, true> : bn_bwd_apply_cf<T, VN, false>;                                          \
        kern<<<(unsigned)(g2.splits * (int64_t)fx.C), 256, 0, st>>>(                                                              \
            (const T *)x->ptr, fx.npitch, early_dz ? nullptr : yp, fy.npitch, early_dz ? zp : (const T *)dy->ptr,                 \
            early_dz ? fdz.npitch : fdy.npitch, (T *)dx->ptr, fdx.npitch, early_dz ? nullptr : zp, fdz.npitch, ws, s, save_mean,  \
            save_invstd, ds, db, M, beta_dx, beta_dz, beta_p, g2);                                                                \
    } while(0)
        if(dt == SAGA_HALF) {
            if(vn == 8) GO(half_t, 8); else GO(half_t, 1);
        } else {
            if(vn == 4) GO(float, 4); else GO(float, 1);
        }
#undef GO
    } else {
        return SAGA_HIP_EUNSUPPORTED;
    }
    SAGA_CHECK_LAUNCH();
    return 0;
}

int saga_hip_bn_bwd_linked(const SagaTensorView *x, const SagaTensorView *g, const SagaTensorView *dx, const float *s,
                           const float *save_mean, const float *save_invstd, float *ds, float *db, float beta_dx,
                           float beta_p, const float *partial, int partial_rows, void *workspace, size_t ws_bytes,
                           saga_stream_t stream)
{
    if(!valid_view(x) || !valid_view(g) || !valid_view(dx) || !s || !save_mean || !save_invstd || !ds || !db || !partial ||
       partial_rows < 1)
        return SAGA_HIP_EINVAL;
    if(!same_dims(x, g) || !same_dims(x, dx))
        return SAGA_HIP_ESHAPE;
    const int dt = x->dtype;
    if((dt != SAGA_HALF && dt != SAGA_FLOAT) || g->dtype != dt || dx->dtype != dt)
        return SAGA_HIP_EUNSUPPORTED;
    CLInfo lx, lg, ldx;
    if(!as_channels_last(x, &lx) || !as_channels_last(g, &lg) || !as_channels_last(dx, &ldx))
        return SAGA_HIP_EUNSUPPORTED;
    const int C = lx.C;
    if(!workspace || ws_bytes < 3 * (size_t)C * sizeof(float))
        return SAGA_HIP_EWORKSPACE;
    hipStream_t st = as_stream(stream);
    float *coef = (float *)workspace;
    const int vn = vec_width(dt, C, {x, g, dx}, {lx.pitch, lg.pitch, ldx.pitch});
    Shape sf;
    if(dt == SAGA_HALF && vn == 8 && self_finalizing(lx.rows, C, partial_rows, true, &sf)) {
        const BwdFin fin = {partial, partial_rows, s, save_invstd, ds, db, (double)lx.rows, beta_p};
        bn_bwd_apply_cl<half_t, 8, false, true><<<dim3(sf.gx, sf.gy), 256, 0, st>>>(
            (const half_t *)x->ptr, lx.pitch, nullptr, 0, (const half_t *)g->ptr, lg.pitch, (half_t *)dx->ptr, ldx.pitch, nullptr, 0,
            save_mean, coef, lx.rows, C, sf.cvb, 0, beta_dx, 0.0f, nullptr, fin);
        SAGA_CHECK_LAUNCH();
        return 0;
    }
    const Shape sh = plan(lx.rows, C / vn, true);
    bn_bwd_finalize<<<C, 256, 0, st>>>(partial, partial_rows, s, save_invstd, ds, db, coef, (double)lx.rows, C, beta_p);
#define GO(T, VN)                                                                                                     \
    bn_bwd_apply_cl<T, VN, false><<<WALK_GRID(8), 256, 0, st>>>((const T *)x->ptr, lx.pitch, nullptr, 0, (const T *)g->ptr,    \
                                                        lg.pitch, (T *)dx->ptr, ldx.pitch, nullptr, 0, save_mean, coef, \
                                                        lx.rows, C, WALK_CVB(8), 0, beta_dx, 0.0f, nullptr)
    if(dt == SAGA_HALF) {
        if(vn == 8) GO(half_t, 8); else GO(half_t, 1);
    } else {
        if(vn == 4) GO(float, 4); else GO(float, 1);
    }
#undef GO
    SAGA_CHECK_LAUNCH();
    return 0;
}

} // extern "C"
