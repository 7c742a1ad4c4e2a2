// fp16 channels-last convolutions for small grids.
//
// The tiled kernels of conv_mfma.hip give a block 256 output pixels x 64 or 128 channels and the whole reduction: a single
// image of ResNet-50's last stages is one block row, two to eight blocks on 256 CUs, each walking up to 144 reduction
// slices one barrier at a time (47 us for a 0.23 GFLOP layer whose filter is 4.7 MB).  Here the tile is as small as 16
// pixels x 16 channels and the wavefronts of a block share the reduction: each walks its own part of it, 32 elements a step
// (v_mfma_f32_16x16x32_f16), through a ring of DEPTH steps of LDS that no other wavefront touches - filled by loads to
// LDS DEPTH - 1 steps ahead, read back in the matrix unit's order, no barrier until the sums of the wavefronts meet at the
// end and leave through the folded batch norm.  The trip through LDS is what makes the loads fast: a load instruction
// fetches 64 bytes of 16 rows with four neighbouring lanes per row, where the operand order would put neighbouring lanes
// on different rows (measured: 73 cycles per kilobyte that way, 34 GB/s and CU).
// Every byte is fetched by every block that needs it, which the caches take while the problem is small; large grids belong
// to the tiled kernels.
#include "stream_f16.hpp"

#include <string.h>
#include <algorithm>
#include <type_traits>

namespace {

constexpr int MAX_CLASSES = 16;
constexpr unsigned OOB = 0x7fffff00u; // beyond every buffer: the load returns zero

// Output pixels whose taps sit at the same distances.  Forward: all of them.  Backward data at stride s: pixels (y, x) with
// the same y mod s and x mod s; inside a class consecutive taps are a fixed distance apart.
struct Class {
    int oy, ox;   // output pixel = class pixel * ostep + (oy, ox)
    int OH, OW;   // the class's grid
    int r0, s0;   // first tap
    int Tr, Ts;   // taps
    int iy0, ix0; // input position of class pixel (0, 0) under its first tap
    int M;        // class pixels over all images
    int block0;   // first block
    int row0;     // first row of sums
};

template <int CLASSES> struct ArgsOf {
    StreamF16 g;
    int istep, ostep, tstep, rstep;
    int nclasses, nblk_q, blocks, KS;
    int q_outer; // blocks that are neighbours share their channels (else their pixels)
    Class cls[CLASSES];
};
typedef ArgsOf<MAX_CLASSES> Args;
typedef ArgsOf<1> Args1;

typedef __attribute__((address_space(3))) void *lds_ptr_t;

// 16 bytes of LDS at a byte address; not an LDS access to the compiler, which would wait for every load to LDS in flight
// in front of it.  The caller waits (lds_wait) before it uses the result.
template <int OFFSET> __device__ __forceinline__ half8_t lds_read(unsigned addr)
{
    half8_t v;
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFFSET));
    return v;
}
template <int N> __device__ __forceinline__ void lds_wait(half8_t (&v)[N])
{
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for(int i = 0; i < N; i++)
        asm volatile("" : "+v"(v[i])); // (results of the reads above, not to be used before the wait)
}

__device__ __forceinline__ int xcd_order(int b, int n)
{
    const int per = n >> 3, rem = n & 7, xcd = b & 7, slot = b >> 3;
    return (xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) + slot;
}

// SUMS: with the per-channel sums (StreamF16::sums)
template <int TM, int TN, int DEPTH, int MAXW, bool SUMS, typename A> __global__ void __launch_bounds__(64 * MAXW) stream_f16_k(A k)
{
    extern __shared__ __attribute__((aligned(16))) float smem[];
    const StreamF16 &g = k.g;
    // as the matrix unit wants its operands, and as the loads fetch them: row lrow, 16-byte piece lkq of its 64.  Rows 4
    // apart fall into the same banks, so they keep their pieces in another order.
    const int tid = threadIdx.x, lane = tid & 63, row = lane & 15, kq = lane >> 4, lrow = lane >> 2;
    const int lkq = (lane & 3) ^ ((lrow >> 2) & 3);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int KS = k.KS, WM = (int)(blockDim.x >> 6) / KS;
    const int wm = wave / KS, ks = wave - wm * KS;
    int b = xcd_order(blockIdx.x, k.blocks), ci = 0;
    while(sizeof(A) > sizeof(Args1) && ci + 1 < k.nclasses && b >= k.cls[ci + 1].block0)
        ci++;
    const Class &c = k.cls[ci];
    b -= c.block0;
    int bm, bq;
    if(k.q_outer) {
        const int nm = (c.M + 16 * TM * WM - 1) / (16 * TM * WM);
        bq = b / nm;
        bm = b - bq * nm;
    } else {
        bm = b / k.nblk_q;
        bq = b - bm * k.nblk_q;
    }
    const int m0 = (bm * WM + wm) * (16 * TM), n0 = bq * (16 * TN);
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void *)g.a, 0, (int)g.a_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc((void *)g.b, 0, (int)g.b_bytes, 0x00020000);

    // byte offset of this lane's 16 bytes of the first tap and first 32 channels (negative outside the image: only valid
    // taps are read), and one bit per tap that falls inside
    int base[TM];
    unsigned long long mask[TM];
#pragma unroll
    for(int i = 0; i < TM; i++) {
        const int m = m0 + 16 * i + lrow;
        const bool ok = m < c.M;
        const int mm = ok ? m : 0;
        const int ox = mm % c.OW, t = mm / c.OW;
        const int oy = t % c.OH, n = t / c.OH;
        const int iy = oy * k.istep + c.iy0, ix = ox * k.istep + c.ix0;
        base[i] = ((n * g.IH + iy) * g.IW + ix) * g.lda * 2 + lkq * 16;
        mask[i] = 0;
        if(ok)
            for(int a = 0; a < c.Tr; a++) {
                const int yy = iy + a * k.tstep;
                if(yy < 0 || yy >= g.IH)
                    continue;
                for(int e = 0; e < c.Ts; e++) {
                    const int xx = ix + e * k.tstep;
                    if(xx >= 0 && xx < g.IW)
                        mask[i] |= 1ull << (a * c.Ts + e);
                }
            }
    }
    int qoff[TN];
#pragma unroll
    for(int t = 0; t < TN; t++) {
        const int n = n0 + 16 * t + lrow;
        qoff[t] = n < g.N ? n * (g.R * g.S * g.C) * 2 + lkq * 16 : -1;
    }

    // the four channels this lane will finish, and what their epilogue needs: requested now, used after the loop
    const int c4 = lane % (TN * 4), nown = n0 + 4 * c4;
    float es[4], eb[4], em[4], ev[4]; // scale, bias, mean, variance of a norm to fold; or scale, bias, mean, 1/std of a linked one
#pragma unroll
    for(int e = 0; e < 4; e++) {
        const int n = nown + e < g.N ? nown + e : 0;
        es[e] = eb[e] = em[e] = ev[e] = 0.0f;
        if(g.bn_s) {
            es[e] = g.bn_s[n];
            eb[e] = g.bn_b[n];
            em[e] = g.bn_m[n];
            ev[e] = g.bn_v[n];
        } else if(SUMS && g.bq_x) {
            em[e] = g.bq_mean[n];
            if(g.bq_relu) {
                es[e] = g.bq_s[n];
                eb[e] = g.bq_b[n];
                ev[e] = g.bq_invstd[n];
            }
        }
    }

    const int S32 = (g.C + 31) / 32, T = c.Tr * c.Ts, total = S32 * T;
    const bool ragged = g.C % 32 != 0;
    const int s_begin = (int)((long long)ks * total / KS), s_end = (int)((long long)(ks + 1) * total / KS);
    int s_next = s_begin, tap = total ? s_begin / S32 : 0, c32 = s_begin - tap * S32;
    int ta = c.Ts ? tap / c.Ts : 0, te = tap - ta * c.Ts;
    unsigned pv[TM], qv[TN];
    auto tap_setup = [&]() {
        const int d = (ta * g.IW + te) * k.tstep * g.lda * 2;
        const int f = ((c.r0 + ta * k.rstep) * g.S + c.s0 + te * k.rstep) * g.C * 2;
#pragma unroll
        for(int i = 0; i < TM; i++)
            pv[i] = (mask[i] >> tap) & 1 ? (unsigned)(base[i] + d) : OOB;
#pragma unroll
        for(int t = 0; t < TN; t++)
            qv[t] = qoff[t] >= 0 ? (unsigned)(qoff[t] + f) : OOB;
    };
    tap_setup();
    constexpr int NL = TM + TN; // load instructions, kilobytes of LDS and operands per step
    char *ring = (char *)smem + wave * (DEPTH * NL * 1024);
    auto load_step = [&](int u) {
        const bool live = s_next < s_end && (!ragged || c32 * 32 + lkq * 8 < g.C);
        char *dst = ring + u * (NL * 1024);
        const int so = c32 * 64;
#pragma unroll
        for(int i = 0; i < TM; i++) {
            const unsigned v = live ? pv[i] : OOB;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_ptr_t)(dst + i * 1024), 16, v, so, 0, 0);
        }
#pragma unroll
        for(int t = 0; t < TN; t++) {
            const unsigned v = live ? qv[t] : OOB;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (lds_ptr_t)(dst + (TM + t) * 1024), 16, v, so, 0, 0);
        }
        if(++c32 == S32) {
            c32 = 0;
            tap++;
            if(++te == c.Ts) {
                te = 0;
                ta++;
            }
            if(s_next + 1 < s_end)
                tap_setup();
        }
        s_next++;
    };
    float4_t acc[TM][TN];
#pragma unroll
    for(int i = 0; i < TM; i++)
#pragma unroll
        for(int t = 0; t < TN; t++)
            acc[i][t] = float4_t{0, 0, 0, 0};
    if(g.bias && ks == 0) // one of the wavefronts that share the reduction starts from it
#pragma unroll
        for(int t = 0; t < TN; t++)
#pragma unroll
            for(int v = 0; v < 4; v++) {
                const int n = n0 + 16 * t + 4 * kq + v;
                const float b = n < g.N ? (float)g.bias[n] : 0.0f;
#pragma unroll
                for(int i = 0; i < TM; i++)
                    acc[i][t][v] = b;
            }
#pragma unroll
    for(int u = 0; u < DEPTH - 1; u++)
        load_step(u);
    const unsigned at = (unsigned)(uintptr_t)(lds_ptr_t)ring + row * 64 + (kq ^ ((row >> 2) & 3)) * 16;
    auto read_step = [&](auto u, half8_t(&f)[NL]) {
        constexpr int U = decltype(u)::value;
        if constexpr(NL > 0) f[0] = lds_read<(U * NL + 0) * 1024>(at);
        if constexpr(NL > 1) f[1] = lds_read<(U * NL + 1) * 1024>(at);
        if constexpr(NL > 2) f[2] = lds_read<(U * NL + 2) * 1024>(at);
        if constexpr(NL > 3) f[3] = lds_read<(U * NL + 3) * 1024>(at);
        if constexpr(NL > 4) f[4] = lds_read<(U * NL + 4) * 1024>(at);
        if constexpr(NL > 5) f[5] = lds_read<(U * NL + 5) * 1024>(at);
        if constexpr(NL > 6) f[6] = lds_read<(U * NL + 6) * 1024>(at);
        if constexpr(NL > 7) f[7] = lds_read<(U * NL + 7) * 1024>(at);
        static_assert(NL <= 8, "operands");
    };
    auto step = [&](auto u, int s) {
        constexpr int U = decltype(u)::value;
        load_step((U + DEPTH - 1) % DEPTH); // into the slot that step s - 1 was read from
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((DEPTH - 1) * NL) : "memory");
        half8_t f[NL];
        read_step(u, f);
        lds_wait(f);
        if(s < s_end) {
#pragma unroll
            for(int i = 0; i < TM; i++)
#pragma unroll
                for(int t = 0; t < TN; t++)
                    acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(f[TM + t], f[i], acc[i][t], 0, 0, 0);
        }
    };
    for(int s = s_begin; s < s_end; s += DEPTH) {
        step(std::integral_constant<int, 0>(), s);
        if constexpr(DEPTH > 1) step(std::integral_constant<int, 1 % DEPTH>(), s + 1);
        if constexpr(DEPTH > 2) step(std::integral_constant<int, 2 % DEPTH>(), s + 2);
        if constexpr(DEPTH > 3) step(std::integral_constant<int, 3 % DEPTH>(), s + 3);
        if constexpr(DEPTH > 4) step(std::integral_constant<int, 4 % DEPTH>(), s + 4);
        if constexpr(DEPTH > 5) step(std::integral_constant<int, 5 % DEPTH>(), s + 5);
        if constexpr(DEPTH > 6) step(std::integral_constant<int, 6 % DEPTH>(), s + 6);
        if constexpr(DEPTH > 7) step(std::integral_constant<int, 7 % DEPTH>(), s + 7);
        static_assert(DEPTH <= 8, "steps");
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // the ring's memory is reused, or the block ends

    // acc[i][t][v]: pixel 16*i + lane%16, channel 16*t + 4*(lane/16) + v
    __syncthreads();
    constexpr int PITCH = TN * 16 + 4, TILE = TM * 16 * PITCH; // floats; rows of a tile fall into different banks
#pragma unroll
    for(int i = 0; i < TM; i++)
#pragma unroll
        for(int t = 0; t < TN; t++)
            *(float4_t *)&smem[wave * TILE + (16 * i + row) * PITCH + 16 * t + 4 * kq] = acc[i][t];
    __syncthreads();
    float sc[4], sh[4];
#pragma unroll
    for(int e = 0; e < 4; e++) {
        sc[e] = es[e] * (SUMS && g.bq_x ? ev[e] : rsqrtf(ev[e] + g.bn_eps));
        sh[e] = SUMS && g.bq_x ? __builtin_fmaf(-em[e], sc[e], eb[e]) : eb[e] - em[e] * sc[e]; // (the forward's own expressions)
    }
    float s1[4] = {0, 0, 0, 0}, s2[4] = {0, 0, 0, 0}; // of this lane's channels: statistics, or sums of a norm's backward
    const bool vec = nown + 4 <= g.N && g.ldo % 4 == 0 && ((uintptr_t)g.out & 7) == 0;
    const bool zvec = vec && g.ldz % 4 == 0 && ((uintptr_t)g.z & 7) == 0;
    for(int e = ks * 64 + lane; e < TM * TN * 64; e += KS * 64) {
        const int px = e / (TN * 4), m = m0 + px;
        const float *s = smem + wm * KS * TILE + px * PITCH + 4 * c4;
        float4_t v = *(const float4_t *)s;
        for(int w = 1; w < KS; w++)
            v += *(const float4_t *)(s + w * TILE);
        if(m >= c.M || nown >= g.N)
            continue;
        const int ox = m % c.OW, t = m / c.OW;
        const int oy = t % c.OH, im = t / c.OH;
        const long long pix = ((long long)im * g.OH + oy * k.ostep + c.oy) * g.OW + ox * k.ostep + c.ox;
        half_t *o = g.out + pix * g.ldo + nown;
        const half_t *z = g.bn_flags & SAGA_BN_ADD ? g.z + pix * g.ldz + nown : nullptr;
        half4_t old = {0, 0, 0, 0}, zz = {0, 0, 0, 0}, xx = {0, 0, 0, 0}, r = {0, 0, 0, 0};
        if(g.beta != 0.0f && vec)
            old = *(const half4_t *)o;
        if(z && zvec)
            zz = *(const half4_t *)z;
        if(SUMS && g.bq_x) // (its callers have made sure of the alignment)
            xx = *(const half4_t *)(g.bq_x + pix * g.bq_ldx + nown);
#pragma unroll
        for(int q = 0; q < 4; q++) {
            if(nown + q >= g.N)
                break;
            float f = g.alpha * v[q];
            if(g.beta != 0.0f)
                f += g.beta * (float)(vec ? old[q] : o[q]);
            if(g.bn_s) {
                f = __builtin_fmaf(f, sc[q], sh[q]);
                if(z)
                    f += (float)(zvec ? zz[q] : z[q]);
                if(g.bn_flags & SAGA_BN_RELU)
                    f = f != f ? f : fmaxf(f, 0.0f);
            }
            r[q] = (half_t)f;
            if(SUMS && g.bq_x) {
                const float xf = (float)xx[q];
                if(g.bq_relu && !((float)(half_t)__builtin_fmaf(xf, sc[q], sh[q]) > 0.0f))
                    r[q] = (half_t)0;
                s1[q] += (float)r[q];
                s2[q] += (float)r[q] * (xf - em[q]);
            } else if(SUMS) {
                s1[q] += (float)r[q];
                s2[q] += (float)r[q] * (float)r[q];
            }
        }
        if(vec) {
            *(half4_t *)o = r;
        } else {
            for(int q = 0; q < 4 && nown + q < g.N; q++)
                o[q] = r[q];
        }
    }
    if constexpr(!SUMS)
        return;
    // lanes with the same channels, then the block's wavefronts
#pragma unroll
    for(int d = TN * 4; d < 64; d *= 2)
#pragma unroll
        for(int q = 0; q < 4; q++) {
            s1[q] += __shfl_xor(s1[q], d, 64);
            s2[q] += __shfl_xor(s2[q], d, 64);
        }
    __syncthreads();
    if(lane < TN * 4)
#pragma unroll
        for(int q = 0; q < 4; q++) {
            smem[(wave * TN * 16 + 4 * c4 + q) * 2] = s1[q];
            smem[(wave * TN * 16 + 4 * c4 + q) * 2 + 1] = s2[q];
        }
    __syncthreads();
    if(tid < TN * 32 && n0 + tid / 2 < g.N) {
        float s = 0.0f;
        for(int w = 0; w < KS * WM; w++)
            s += smem[w * TN * 32 + tid];
        g.sums[((long long)(c.row0 + bm) * g.N + n0) * 2 + tid] = s;
    }
}

struct Config {
    int tm, tn, ks, wm;
};

// Tile (16*tm pixels x 16*tn channels per wavefront) and wavefronts along the reduction (ks) and the pixels (wm) for a
// problem of `tiles` 16x16 tiles and `steps` reduction steps of 32; tm = 0: a matter for the tiled kernels.  Small tiles
// fill the chip, larger ones fetch less per multiplication, and a wavefront should walk more steps than its ring holds.
// Measured (us; tm,tn,ks,wm; the tiled kernel last; launch included):
//   1x14x14 3x3 256->256    tiles  208 steps  72   1,1,4,1  7.4  1,1,8,1  7.6  2,2,8,1  9.2   28
//   1x7x7   3x3 512->512            128       144  1,1,8,1  8.5  1,1,4,1  9.1  2,2,8,1 11.2   47
//   1x28x28 1x1 512->128            392        16  1,1,2,2  4.8  2,2,4,1  5.1  1,1,4,1  5.6    8.9
//   1x14x14 1x1 256->1024           832         8  1,1,1,4  4.9  2,2,4,1  5.3                  6.7
//   1x56x56 3x3 64->64              784        18  2,2,4,1  7.1  2,2,8,1  7.4  1,1,1,4  7.7   11
//   4x14x14 3x3 256->256            784        72  2,2,8,1  9.8  2,2,4,1 10.1  4,2,8,1 11.5   28
//   4x28x28 3x3 128->128           1568        36  2,2,4,1 10.1  4,2,8,1 10.4  2,2,2,2 10.7   18
//   16x7x7  3x3 512->512           1568       144  4,2,8,1 18.1  2,2,4,1 21.5  2,2,2,2 22.9   48
//   16x14x14 1x1 1024->256         3136        32  2,2,2,2 11.0  4,4,4,1 11.7  4,2,4,1 11.9   14
//   16x14x14 3x3 256->256          3136        72  4,4,4,1 18.1  2,2,2,2 18.4  4,2,4,1 20.0   28
//   32x14x14 3x3 256->256          6272        72  4,4,2,2 27.9                               28.5
//   4x14x14 1x1 256->1024          3136         8  2,2,2,2  7.2                                6.9
// Beyond these the sums of a tile are better shared by several blocks of the tiled kernel (42x42 3x3 1024->512: 35 against
// 48 us here and 96 alone).
Config choose(long long tiles, long long steps, int N)
{
    if(tiles > 3600 || (steps >= 200 && tiles >= 1500) || (steps >= 128 && tiles > 3300))
        return {0, 0, 0, 0};
    if(tiles <= 640) {
        if(steps < 8)
            return {0, 0, 0, 0};
        return steps >= 100 ? Config{1, 1, 8, 1} : steps >= 24 ? Config{1, 1, 4, 1} : steps >= 12 ? Config{1, 1, 2, 2} : Config{1, 1, 1, 4};
    }
    if(tiles <= 2048) {
        if(steps < 12)
            return steps >= 8 && tiles <= 900 ? Config{1, 1, 1, 4} : Config{0, 0, 0, 0};
        if(steps >= 100 && tiles > 1200)
            return {4, 2, 8, 1};
        return {2, 2, steps >= 64 && tiles <= 900 ? 8 : 4, 1};
    }
    // (wide tiles only for channels that fill them: 5x5 160->32 at 57x17x17 25 against 51 us, the tiled kernel 27.  Its tiles of
    // 64 channels are enough blocks for narrow layers: 5x5 64->16 at 49x30x30 24 against 29, 48->40 at 7x50x50 26 against 30)
    if(steps >= 64)
        return N > 32 ? Config{4, 4, 4, 1} : Config{4, 2, 4, 1};
    return steps >= 16 && N > (steps >= 32 ? 64 : 16) ? Config{2, 2, 2, 2} : Config{0, 0, 0, 0};
}

Config config_of(const StreamF16 &g)
{
    const int s = g.bwd ? g.stride : 1;
    const long long pixels = (long long)g.batch * ((g.OH + s - 1) / s) * ((g.OW + s - 1) / s) * s * s;
    const long long taps = ((g.R + s - 1) / s) * ((g.S + s - 1) / s);
    return choose((pixels + 15) / 16 * ((g.N + 15) / 16), taps * ((g.C + 31) / 32), g.N);
}

int gcd(int a, int b) { return b ? gcd(b, a % b) : a; }

bool classes(Args &a)
{
    const StreamF16 &g = a.g;
    const int s = g.bwd ? g.stride : 1;
    if(s * s > MAX_CLASSES)
        return false;
    a.nclasses = s * s;
    a.istep = g.bwd ? 1 : g.stride;
    a.ostep = s;
    const int q = gcd(s, g.dil);
    a.rstep = s / q;
    a.tstep = g.bwd ? -g.dil / q : g.dil;
    for(int i = 0; i < a.nclasses; i++) {
        Class &c = a.cls[i];
        c.oy = i / s;
        c.ox = i % s;
        c.OH = (g.OH - c.oy + s - 1) / s;
        c.OW = (g.OW - c.ox + s - 1) / s;
        auto axis = [&](int o, int taps, int &first, int &n, int &pos) {
            for(first = 0; first < a.rstep && (o + g.pad - first * g.dil) % s; first++)
                ;
            if(!g.bwd) {
                n = taps;
                pos = -g.pad;
                return;
            }
            n = first < a.rstep && first < taps ? (taps - first + a.rstep - 1) / a.rstep : 0;
            pos = n ? (o + g.pad - first * g.dil) / s : 0; // divides
        };
        axis(c.oy, g.R, c.r0, c.Tr, c.iy0);
        axis(c.ox, g.S, c.s0, c.Ts, c.ix0);
        if(!c.Tr || !c.Ts)
            c.Tr = c.Ts = 0;
        if(c.Tr * c.Ts > 64)
            return false;
        c.M = g.batch * c.OH * c.OW;
    }
    return true;
}

template <bool SUMS, typename A> int launch_as(const A &k, const Config &cf, hipStream_t st)
{
    const int threads = 64 * cf.ks * cf.wm;
#define GO(TM, TN, DEPTH, MAXW)                                                                                             \
    do {                                                                                                                    \
        auto kern = stream_f16_k<TM, TN, DEPTH, MAXW, SUMS, A>;                                                                  \
        constexpr size_t wave_lds = std::max(DEPTH * (TM + TN) * 1024, TM * 16 * (TN * 16 + 4) * 4);                         \
        static const hipError_t attr = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize,   \
                                                           MAXW * wave_lds);                                                \
        if(attr != hipSuccess)                                                                                              \
            return (int)attr;                                                                                               \
        kern<<<k.blocks, threads, wave_lds *(threads / 64), st>>>(k);                                                       \
    } while(0)
    if(cf.tm == 4 && cf.tn == 4)
        GO(4, 4, 3, 4);
    else if(cf.tm == 4)
        GO(4, 2, 3, 8);
    else if(cf.tm == 2)
        GO(2, 2, 4, 8);
    else
        GO(1, 1, 8, 8);
#undef GO
    SAGA_CHECK_LAUNCH();
    return 0;
}

} // namespace

bool stream_f16_wanted(const StreamF16 &g) { return config_of(g).tm > 0; }

int stream_f16_sum_rows(const StreamF16 &g)
{
    const Config cf = config_of(g);
    const int s = g.bwd ? g.stride : 1;
    const long long M = (long long)g.batch * ((g.OH + s - 1) / s) * ((g.OW + s - 1) / s);
    return cf.tm ? (int)((M + 16 * cf.tm * cf.wm - 1) / (16 * cf.tm * cf.wm)) * s * s : 0;
}

int stream_f16_launch(const StreamF16 &g, hipStream_t st, int *sum_rows)
{
    Args k = {};
    k.g = g;
    if(g.C % 8 || g.lda % 8 || !g.a_bytes || !g.b_bytes || !classes(k))
        return SAGA_HIP_EUNSUPPORTED;
    const Config cf = config_of(g);
    if(!cf.tm)
        return SAGA_HIP_EUNSUPPORTED;
    k.KS = cf.ks;
    k.nblk_q = (g.N + 16 * cf.tn - 1) / (16 * cf.tn);
    // the larger operand is the one that each die should fetch once
    k.q_outer = (long long)g.N * g.R * g.S > (long long)g.batch * g.IH * g.IW;
    long long blocks = 0;
    int rows = 0;
    for(int i = 0; i < k.nclasses; i++) {
        k.cls[i].block0 = (int)blocks;
        k.cls[i].row0 = rows;
        rows += (k.cls[i].M + 16 * cf.tm * cf.wm - 1) / (16 * cf.tm * cf.wm);
        blocks = (long long)rows * k.nblk_q;
    }
    if(sum_rows)
        *sum_rows = rows;
    if(blocks > 0x7fffffff)
        return SAGA_HIP_EUNSUPPORTED;
    k.blocks = (int)blocks;
    if(k.nclasses > 1)
        return g.sums ? launch_as<true>(k, cf, st) : launch_as<false>(k, cf, st);
    Args1 one;
    memcpy((void *)&one, &k, sizeof(one)); // the same members up to the first class
    return g.sums ? launch_as<true>(one, cf, st) : launch_as<false>(one, cf, st);
}
