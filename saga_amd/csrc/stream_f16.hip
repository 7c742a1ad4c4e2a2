// fp16 channels-last convolutions for small grids.
//
// The tiled kernels of conv_mfma.hip give a block 256 output pixels x 64 or 128 channels and the whole reduction: a single
// image of ResNet-50's last stages is one block row, two to eight blocks on 256 CUs, each walking up to 144 reduction
// slices one barrier at a time (47 us for a 0.23 GFLOP layer whose filter is 4.7 MB).  Here the tile is as small as 16
// pixels x 16 channels and the wavefronts of a block share the reduction: each walks its own part of it, 32 or 64 elements a
// step (v_mfma_f32_16x16x32_f16), through a ring of DEPTH steps of LDS that no other wavefront touches - filled by loads to
// LDS DEPTH - 1 steps ahead, read back in the matrix unit's order, no barrier until the sums of the wavefronts meet at the
// end and leave through the folded batch norm.  The trip through LDS is what makes the loads fast: a load instruction
// fetches 64 bytes of 16 rows with four neighbouring lanes per row, or 128 of 8 with eight, where the operand order would put neighbouring lanes
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

// n / d for 0 <= n < 2^31 without a division
struct Div {
    unsigned mul, shift;
};

Div div_by(unsigned d)
{
    Div v = {1, 0};
    while((1u << v.shift) < d)
        v.shift++;
    v.mul = (unsigned)((((unsigned long long)((1u << v.shift) - d)) << 32) / d) + 1;
    return v;
}

__device__ __forceinline__ int divide(int n, Div d) { return (int)((__umulhi((unsigned)n, d.mul) + (unsigned)n) >> d.shift); }

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
    int nm;       // blocks along the pixels
    Div by_OH, by_OW, by_Ts, by_nm;
};

template <int CLASSES> struct ArgsOf {
    StreamF16 g;
    int istep, ostep, tstep, rstep;
    int nclasses, nblk_q, blocks;
    int ks_log2, WM, S; // wavefronts along the reduction and the pixels; steps per tap
    Div by_q, by_S;
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
// tiles I to N - 1 of SIZE bytes each
template <int SIZE, int I = 0, int N> __device__ __forceinline__ void lds_read_tiles(half8_t (&v)[N], unsigned addr)
{
    if constexpr(I < N) {
        v[I] = lds_read<I * SIZE>(addr);
        lds_read_tiles<SIZE, I + 1>(v, addr);
    }
}
template <int U, int N> __device__ __forceinline__ void lds_wait(half8_t (&v)[U][N])
{
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for(int u = 0; u < U; u++)
#pragma unroll
        for(int i = 0; i < N; i++)
            asm volatile("" : "+v"(v[u][i])); // (results of the reads above, not to be used before the wait)
}

// LDS of a wavefront: the ring of DEPTH steps, or for DEPTH = 0 of RING tiles, then its sums in the same place
constexpr int RING = 9;
template <int TM, int TN, int U, int DEPTH> constexpr int wave_lds()
{
    return std::max((DEPTH ? DEPTH * (TM + TN) : RING) * U * 1024, TM * 16 * (TN * 16 + 4) * 4);
}

typedef unsigned uint2_t __attribute__((ext_vector_type(2)));
typedef unsigned uint4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer(const void *p, unsigned bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc((void *)p, 0, p ? (int)bytes : 0, 0x00020000);
}

// Four channels of a tensor from byte offset `at` (OOB: none), in one access - at any address of a half, the hardware splits what crosses
// a line - or, where a block's channels end inside four, one by one, `n` of them inside the row.
__device__ __forceinline__ half4_t load4(__amdgpu_buffer_rsrc_t r, unsigned at, bool vec, int n)
{
    if(vec)
        return __builtin_bit_cast(half4_t, (uint2_t)__builtin_amdgcn_raw_buffer_load_b64(r, at, 0, 0));
    half4_t v;
#pragma unroll
    for(int q = 0; q < 4; q++)
        v[q] = __builtin_bit_cast(half_t, (unsigned short)__builtin_amdgcn_raw_buffer_load_b16(r, q < n ? at + 2 * q : OOB, 0, 0));
    return v;
}
__device__ __forceinline__ void store4(__amdgpu_buffer_rsrc_t r, unsigned at, bool vec, int n, half4_t v)
{
    if(vec) {
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(uint2_t, v), r, at, 0, 0);
        return;
    }
#pragma unroll
    for(int q = 0; q < 4; q++) {
        const half_t one = v[q]; // (the cast of a vector's element takes the first)
        __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(unsigned short, one), r, q < n ? at + 2 * q : OOB, 0, 0);
    }
}

// A launch takes a few microseconds, and most of them are trips to memory in a row: the arguments, the code (every 64 bytes
// are a miss the first time a CU meets them), the operands, what the epilogue reads.  So the lines of the arguments are all
// touched first; the epilogue's operands are requested in front of the reduction, through buffer loads that need no branch
// (behind a branch the compiler waits for each before the next); divisions are multiplications; tap bits are kept by row and
// column; a step is the same code for all taps, its loop inside the loop over the taps.
// One image of 14x14 pixels, us in the kernel, against the same tiles with the ring unrolled (11 KB of code): 1x1 256->1024
// 4.8 -> 3.0 (now 0.6 setup, 0.8 filling the ring, 0.7 the rest of the reduction, 0.2 the sum of the wavefronts, 0.5
// epilogue), 1x1 1024->256 4.7 -> 3.3, 3x3 256->256 7.1 -> 4.6; from the end of a launch to the next it is 1.4.
// SUMS: with the per-channel sums (StreamF16::sums)
// U: a step takes 32 * U channels.  With 32, two steps share the cache lines of their rows, and what the other wavefronts load
// between them is more than a CU's cache holds: every line came from L2 twice, and that is what bounds the larger problems (1x21x21
// 3x3 1024->1024: 5.6 M lines read for 5.9 M pieces of 64 bytes).  With 64 an instruction takes whole lines.  us, 32 / 64, the best tile of
// each: 1x21x21 3x3 1024->1024 30.0 / 21.1, 1x42x42 3x3 512->512 25.2 / 17.8, 23x13x13 3x3 256->256 15.5 / 12.5, 1x7x7 3x3 512->512
// 7.0 / 6.4, 4x14x14 3x3 512->512 at stride 2 10.2 / 9.2; with few steps to a wavefront (1x28x28 3x3 128->128) equal.
// DEPTH = 0: eight wavefronts with tiles of 64 pixels x 32 channels have no room for two steps of 64 channels, but for one and a half.
// Their ring holds single operands of 16 rows, each of which leaves room for the one nine later as soon as it is in registers.
template <int TM, int TN, int U, int DEPTH, int MAXW, bool SUMS, typename A> __global__ void __launch_bounds__(64 * MAXW) stream_f16_k(A k)
{
    extern __shared__ __attribute__((aligned(16))) float smem[];
    constexpr bool ONE = sizeof(A) == sizeof(Args1); // one class: class pixels are output pixels
    const StreamF16 &g = k.g;
    {
        const __attribute__((address_space(4))) int *line = (const __attribute__((address_space(4))) int *)__builtin_amdgcn_kernarg_segment_ptr();
        static_assert(sizeof(Args1) > 5 * 64, "arguments");
        asm volatile("" ::"s"(line[0]), "s"(line[16]), "s"(line[32]), "s"(line[48]), "s"(line[64]), "s"(line[80]));
    }
    // as the matrix unit wants its operands (row, kq), and as the loads fetch them: 16 / U rows by an instruction, each lane the
    // 16-byte piece lkq of the 64 * U bytes of a row.  Rows 4 / U apart fall into the same banks, so they keep their pieces
    // in another order; that of the second half of 16 rows is the first's with bit 2 flipped.
    const int tid = threadIdx.x, lane = tid & 63, row = lane & 15, kq = lane >> 4;
    auto lrow = [&](int i) { return 16 / U * i + lane / (4 * U); };
    auto lkq = [&](int i) { return U == 1 ? (lane & 3) ^ (lane >> 4) : (lane & 7) ^ (lane >> 4) ^ 4 * (i & 1); };
    auto spot = [&](int u) { return row * (64 * U) + ((4 * u + kq) ^ (row * U >> 2)) * 16; };
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int KS = 1 << k.ks_log2, wm = wave >> k.ks_log2, ks = wave & (KS - 1);
    int b = xcd_remap(blockIdx.x, k.blocks), ci = 0;
    while(!ONE && ci + 1 < k.nclasses && b >= k.cls[ci + 1].block0)
        ci++;
    const Class &c = k.cls[ci];
    b -= c.block0;
    const int outer = divide(b, k.q_outer ? c.by_nm : k.by_q), inner = b - outer * (k.q_outer ? c.nm : k.nblk_q);
    const int bm = k.q_outer ? inner : outer, bq = k.q_outer ? outer : inner;
    const int m0 = (bm * k.WM + wm) * (16 * TM), n0 = bq * (16 * TN);
    const __amdgpu_buffer_rsrc_t ra = buffer(g.a, g.a_bytes), rb = buffer(g.b, g.b_bytes);

    // byte offset of this lane's 16 bytes of the first tap and first 32 channels (negative outside the image: only valid
    // taps are read), and one bit per row and column of taps that falls inside
    constexpr int LM = TM * U, LN = TN * U; // load instructions of a step
    int base[LM], iy[LM], ix[LM];
    unsigned rows[LM], cols[LM];
#pragma unroll
    for(int i = 0; i < LM; i++) {
        const int m = m0 + lrow(i);
        const bool ok = m < c.M;
        const int mm = ok ? m : 0;
        const int t = divide(mm, c.by_OW), ox = mm - t * c.OW;
        const int n = divide(t, c.by_OH), oy = t - n * c.OH;
        iy[i] = oy * k.istep + c.iy0;
        ix[i] = ox * k.istep + c.ix0;
        base[i] = ((n * g.IH + iy[i]) * g.IW + ix[i]) * g.lda * 2 + lkq(i) * 16;
        rows[i] = cols[i] = 0;
        iy[i] = ok ? iy[i] : 0x40000000; // (no row of the image)
    }
#pragma unroll 1
    for(int a = 0; a < c.Tr; a++)
#pragma unroll
        for(int i = 0; i < LM; i++)
            rows[i] |= (unsigned)(iy[i] + a * k.tstep) < (unsigned)g.IH ? 1u << a : 0u;
#pragma unroll 1
    for(int a = 0; a < c.Ts; a++)
#pragma unroll
        for(int i = 0; i < LM; i++)
            cols[i] |= (unsigned)(ix[i] + a * k.tstep) < (unsigned)g.IW ? 1u << a : 0u;
    int qoff[LN];
#pragma unroll
    for(int t = 0; t < LN; t++) {
        const int n = n0 + lrow(t);
        qoff[t] = n < g.N ? n * (g.R * g.S * g.C) * 2 + lkq(t) * 16 : -1;
    }

    // the four channels this lane will finish, and what their epilogue needs: requested now, used after the loop
    const int c4 = lane % (TN * 4), nown = n0 + 4 * c4;
    auto channels = [&](const float *p) {
        return __builtin_bit_cast(float4_t, (uint4_t)__builtin_amdgcn_raw_buffer_load_b128(buffer(p, 4u * g.N), 4 * nown, 0, 0));
    };
    // scale, bias, mean, variance of a norm to fold; or scale, bias, mean, 1/std of a linked one
    const bool linked = SUMS && g.bq_x;
    const float4_t es = channels(linked ? g.bq_s : g.bn_s), em = channels(linked ? g.bq_mean : g.bn_m);
    const float4_t ev = channels(linked ? g.bq_invstd : g.bn_v), eb = channels(linked ? g.bq_b : g.bn_b);
    half4_t bias = {0, 0, 0, 0};
    if(g.bias)
        bias = load4(buffer(g.bias, 2u * g.N), 2 * nown, false, g.N - nown);
    // and of the first (mostly the only) pixel: what it adds to (beta), its residual, the norm's input
    const bool vec = (g.N & 3) == 0 || n0 + 16 * TN <= g.N;
    const bool with_z = g.bn_flags & SAGA_BN_ADD;
    const __amdgpu_buffer_rsrc_t ro = buffer(g.out, g.out_bytes), rz = buffer(with_z ? g.z : nullptr, g.z_bytes);
    const __amdgpu_buffer_rsrc_t rwas = buffer(g.beta != 0.0f ? g.out : nullptr, g.out_bytes);
    half4_t old, zz, xx;
    auto pixel = [&](int e) { // -1: none
        const int m = m0 + e / (TN * 4);
        if(ONE)
            return e < TM * TN * 64 && m < c.M && nown < g.N ? m : -1;
        const int t = divide(m, c.by_OW), ox = m - t * c.OW;
        const int im = divide(t, c.by_OH), oy = t - im * c.OH;
        return e < TM * TN * 64 && m < c.M && nown < g.N ? (im * g.OH + oy * k.ostep + c.oy) * g.OW + ox * k.ostep + c.ox : -1;
    };
    auto request = [&](int pix) {
        old = load4(rwas, pix >= 0 ? (unsigned)(pix * g.ldo + nown) * 2 : OOB, vec, g.N - nown);
        zz = load4(rz, pix >= 0 ? (unsigned)(pix * g.ldz + nown) * 2 : OOB, vec, g.N - nown);
        if(SUMS) // (its callers have made sure of the alignment)
            xx = load4(buffer(g.bq_x, g.bq_bytes), pix >= 0 ? (unsigned)(pix * g.bq_ldx + nown) * 2 : OOB, true, 4);
    };
    int e = ks * 64 + lane, pix = pixel(e);
    request(pix);

    const int S = k.S, total = S * c.Tr * c.Ts;
    const bool last_ok = (S - 1) * 32 + lkq(0) * 8 < g.C;
    const int cut = U == 1 && g.C % 32 ? (S - 1) * 64 : -1; // where only some of the 32 channels are there
    const int s_begin = (ks * total) >> k.ks_log2, steps = ((ks * total + total) >> k.ks_log2) - s_begin;
    int tap = divide(s_begin, k.by_S), c0 = s_begin - tap * S;
    int ta = divide(tap, c.by_Ts), te = tap - ta * c.Ts;
    constexpr int NL = LM + LN; // load instructions, kilobytes of LDS and operands per step
    char *ring = (char *)smem + wave * wave_lds<TM, TN, U, DEPTH>();
    const unsigned at = (unsigned)(uintptr_t)(lds_ptr_t)ring;
    auto load_to_lds = [](__amdgpu_buffer_rsrc_t r, char *dst, unsigned v, int at) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr_t)dst, 16, v, at, 0, 0);
    };
    float4_t acc[TM][TN];
#pragma unroll
    for(int i = 0; i < TM; i++)
#pragma unroll
        for(int t = 0; t < TN; t++)
            acc[i][t] = float4_t{0, 0, 0, 0};
    int fill = 0, drain = 0;
    auto consume = [&]() {
        half8_t f[U][TM + TN];
#pragma unroll
        for(int u = 0; u < U; u++)
            lds_read_tiles<U * 1024>(f[u], at + drain + spot(u));
        drain = drain == (DEPTH - 1) * NL * 1024 ? 0 : drain + NL * 1024;
        lds_wait(f); // before the next step loads into this slot
#pragma unroll
        for(int u = 0; u < U; u++)
#pragma unroll
            for(int i = 0; i < TM; i++)
#pragma unroll
                for(int t = 0; t < TN; t++)
                    acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(f[u][TM + t], f[u][i], acc[i][t], 0, 0, 0);
    };
    // operand v of a step: of the channels, then of the pixels
    half8_t fn[TN][U];
    auto take = [&](int v) {
        half8_t f[U][1];
#pragma unroll
        for(int u = 0; u < U; u++)
            f[u][0] = lds_read<0>(at + drain + spot(u));
        drain = drain == (RING - 1) * U * 1024 ? 0 : drain + U * 1024;
        lds_wait(f); // before its place is loaded again
#pragma unroll
        for(int u = 0; u < U; u++)
#pragma unroll
            for(int t = 0; t < TN; t++)
                if(v == t)
                    fn[t][u] = f[u][0];
                else if(v >= TN)
                    acc[v - TN][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fn[t][u], f[u][0], acc[v - TN][t], 0, 0, 0);
    };
    int s = 0; // steps requested
#pragma unroll 1
    while(s < steps) {
        const int d = (ta * g.IW + te) * k.tstep * g.lda * 2;
        const int f = ((c.r0 + ta * k.rstep) * g.S + c.s0 + te * k.rstep) * g.C * 2;
        unsigned pv[LM], qv[LN];
#pragma unroll
        for(int i = 0; i < LM; i++)
            pv[i] = (rows[i] >> ta) & (cols[i] >> te) & 1 ? (unsigned)(base[i] + d) : OOB;
#pragma unroll
        for(int t = 0; t < LN; t++)
            qv[t] = qoff[t] >= 0 ? (unsigned)(qoff[t] + f) : OOB;
        const int until = std::min(s + S - c0, steps);
        int so = c0 * (64 * U);
#pragma unroll 1
        do {
            if(so == cut) { // (the tap's last step)
#pragma unroll
                for(int i = 0; i < LM; i++)
                    pv[i] = last_ok ? pv[i] : OOB;
#pragma unroll
                for(int t = 0; t < LN; t++)
                    qv[t] = last_ok ? qv[t] : OOB;
            }
            if constexpr(DEPTH == 0) {
#pragma unroll
                for(int v = 0; v < TM + TN; v++) {
#pragma unroll
                    for(int u = 0; u < U; u++)
                        load_to_lds(v < TN ? rb : ra, ring + fill + u * 1024, v < TN ? qv[v * U + u] : pv[(v - TN) * U + u], so);
                    fill = fill == (RING - 1) * U * 1024 ? 0 : fill + U * 1024;
                    constexpr int BEHIND = RING - 1, PER = TM + TN; // operands requested behind the one to take
                    if(s * PER + v >= BEHIND) {
                        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(BEHIND * U) : "memory");
                        take((v + 2 * PER - BEHIND) % PER);
                    }
                }
                so += 64 * U;
                continue;
            }
#pragma unroll
            for(int i = 0; i < LM; i++)
                load_to_lds(ra, ring + fill + i * 1024, pv[i], so);
#pragma unroll
            for(int t = 0; t < LN; t++)
                load_to_lds(rb, ring + fill + (LM + t) * 1024, qv[t], so);
            fill = fill == (DEPTH - 1) * NL * 1024 ? 0 : fill + NL * 1024;
            so += 64 * U;
            if(s >= DEPTH - 1) {
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"((DEPTH - 1) * NL) : "memory");
                consume();
            }
        } while(++s < until);
        c0 = 0;
        if(++te == c.Ts) {
            te = 0;
            ta++;
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if constexpr(DEPTH == 0) {
        static_assert(DEPTH || (RING > TM + TN && RING - 1 <= 2 * (TM + TN)), "the last operands of a step and all of the next");
#pragma unroll
        for(int v = 2 * (TM + TN) - (RING - 1); v < TM + TN; v++)
            if(steps > 1)
                take(v);
#pragma unroll
        for(int v = 0; v < TM + TN; v++)
            if(steps > 0)
                take(v);
    } else {
#pragma unroll 1
        for(int u = std::min(steps, DEPTH - 1); u > 0; u--)
            consume();
    }

    // acc[i][t][v]: pixel 16*i + lane%16, channel 16*t + 4*(lane/16) + v
    constexpr int PITCH = TN * 16 + 4, WAVE = wave_lds<TM, TN, U, DEPTH>() / 4; // floats; rows of a tile fall into different banks
#pragma unroll
    for(int i = 0; i < TM; i++)
#pragma unroll
        for(int t = 0; t < TN; t++)
            *(float4_t *)&smem[wave * WAVE + (16 * i + row) * PITCH + 16 * t + 4 * kq] = acc[i][t];
    float4_t sc, sh;
#pragma unroll
    for(int q = 0; q < 4; q++) {
        sc[q] = es[q] * (linked ? ev[q] : rsqrtf(ev[q] + g.bn_eps));
        sh[q] = linked ? __builtin_fmaf(-em[q], sc[q], eb[q]) : eb[q] - em[q] * sc[q]; // (the forward's own expressions)
    }
    __syncthreads();
    float s1[4] = {0, 0, 0, 0}, s2[4] = {0, 0, 0, 0}; // of this lane's channels: statistics, or sums of a norm's backward
#pragma unroll 1
    for(; e < TM * TN * 64;) {
        const float *part = smem + wm * KS * WAVE + e / (TN * 4) * PITCH + 4 * c4;
        float4_t v = *(const float4_t *)part;
        if(KS >= 2)
            v += *(const float4_t *)(part + WAVE);
        if(KS >= 4) {
            const float4_t v2 = *(const float4_t *)(part + 2 * WAVE), v3 = *(const float4_t *)(part + 3 * WAVE);
            v = v + v2 + v3;
        }
        if(KS >= 8) {
            const float4_t v4 = *(const float4_t *)(part + 4 * WAVE), v5 = *(const float4_t *)(part + 5 * WAVE);
            const float4_t v6 = *(const float4_t *)(part + 6 * WAVE), v7 = *(const float4_t *)(part + 7 * WAVE);
            v = v + v4 + v5 + v6 + v7;
        }
        const half4_t was = old, res = zz, in = xx;
        const int here = pix;
        e += KS * 64;
        if constexpr(TM * TN > 1) {
            pix = pixel(e);
            request(pix);
        }
        v *= g.alpha;
        if(g.bias)
            v += __builtin_convertvector(bias, float4_t);
        if(g.beta != 0.0f)
            v += g.beta * __builtin_convertvector(was, float4_t);
        if(g.bn_s) {
#pragma unroll
            for(int q = 0; q < 4; q++)
                v[q] = __builtin_fmaf(v[q], sc[q], sh[q]);
            if(with_z)
                v += __builtin_convertvector(res, float4_t);
            if(g.bn_flags & SAGA_BN_RELU)
#pragma unroll
                for(int q = 0; q < 4; q++)
                    v[q] = v[q] != v[q] ? v[q] : fmaxf(v[q], 0.0f);
        }
        half4_t r = __builtin_convertvector(v, half4_t);
        if(SUMS && here >= 0) {
            if(linked) {
#pragma unroll
                for(int q = 0; q < 4; q++) {
                    const float xf = (float)in[q];
                    if(g.bq_relu && !((float)(half_t)__builtin_fmaf(xf, sc[q], sh[q]) > 0.0f))
                        r[q] = (half_t)0;
                    s1[q] += (float)r[q];
                    s2[q] += (float)r[q] * (xf - em[q]);
                }
            } else {
#pragma unroll
                for(int q = 0; q < 4; q++) {
                    s1[q] += (float)r[q];
                    s2[q] += (float)r[q] * (float)r[q];
                }
            }
        }
        store4(ro, here >= 0 ? (unsigned)(here * g.ldo + nown) * 2 : OOB, vec, g.N - nown, r);
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
        for(int w = 0; w < KS * k.WM; w++)
            s += smem[w * TN * 32 + tid];
        g.sums[((long long)(c.row0 + bm) * g.N + n0) * 2 + tid] = s;
    }
}

struct Config {
    int tm, tn, u, ks, wm;
};

// Tile (16*tm pixels x 16*tn channels per wavefront), 32*u channels to a step (64 only where they divide C) and wavefronts along the
// reduction (ks) and the pixels (wm) by what they cost: start + steps of a wavefront * (step + more * rounds) + round * rounds, where a round is a block on every CU.
// The numbers are fitted to 420 problems (1 to 90 images of 7x7 to 150x150 pixels, 8 to 2048 channels either way, filters
// of 1 to 5; those of u = 2 to 180 of 64 to 2048 channels) at each of the tiles, launched one behind the other with filters that are not
// in the cache: 8 % off on average, and the choice 4 % (2 % with u = 2 in it) slower than the best of everything at each problem
// (lines drawn by tiles and steps, which stood here before: 16 %).  Left out, as no choice got better with them: u = 2 at 1x1 tiles
// without a split or of 8, 2x2 of 2x2 and of 8, 4x2 of 2x2.  us, drawn lines -> fitted costs of u = 1, of which the tiled kernels
// where they took it:
//   1x56x56 3x3 64->64 and below  as before              23x13x13 3x3 256->256   27.1 -> 15.3 (tiled before)
//   2x28x28 1x1 128->512     6.0 -> 5.0 (tiled before)  16x28x28 3x3 128->128   18.8 -> 14.1 (tiled before)
//   1x28x28 1x1 128->512     5.8 -> 4.1 (tiled before)  512x8x8  3x3 64->64     18.6 -> 10.7 (tiled before)
//   4x14x14 3x3 512->512 /2 12.7 -> 9.9                 49x30x30 5x5 64->16     23.1 -> 15.3 (tiled before)
struct Cost {
    Config c;
    float start, step, more, round;
};
constexpr Cost COSTS[] = {
    {{1, 1, 1, 1, 4}, 3.48f, 0.053f, 0.046f, 0.31f},
    {{1, 1, 1, 4, 1}, 3.33f, 0.028f, 0.079f, 0.29f},
    {{1, 1, 1, 8, 1}, 1.97f, 0.046f, 0.174f, 1.70f},
    {{2, 2, 1, 2, 2}, 3.63f, 0.048f, 0.141f, 0.66f},
    {{2, 2, 1, 4, 1}, 3.31f, 0.054f, 0.167f, 0.48f},
    {{4, 2, 1, 2, 2}, 4.85f, -0.057f, 0.345f, 0.46f},
    {{4, 2, 1, 8, 1}, 1.58f, 0.051f, 0.572f, 2.63f},
    {{4, 4, 1, 2, 2}, 2.09f, -0.083f, 0.463f, 5.29f},
    {{4, 4, 1, 4, 1}, 1.49f, -0.008f, 0.439f, 4.34f},
    {{1, 1, 2, 4, 1}, 2.96f, 0.016f, 0.134f, 0.45f},
    {{2, 2, 2, 4, 1}, 3.32f, 0.044f, 0.256f, 0.62f},
    {{4, 2, 2, 8, 1}, 1.41f, 0.000f, 0.878f, 3.89f},
    {{4, 4, 2, 2, 2}, 3.48f, 0.000f, 0.554f, 5.20f},
    {{4, 4, 2, 4, 1}, 4.45f, 0.000f, 0.594f, 2.50f},
};

int split_over(long long a, long long b) { return (int)((a + b - 1) / b); }

// the tiled kernels: 256 pixels x 64 or 128 channels per block, the reduction of a tile split over k blocks where that pays
float tiled_us(long long pixels, int steps, int N)
{
    const int bn = N <= 64 ? 64 : 128;
    const long long tiles = (pixels + 255) / 256 * split_over(N, bn);
    const int k = N % 8 == 0 ? conv_tile_split(tiles, bn, steps) : 1, L = split_over(steps, k), rounds = split_over(tiles, 256);
    if(k > 1)
        return 13.3f + 0.47f * L + (bn == 64 ? 1.0f : 8.0f) * (tiles * k) / 256.0f;
    if(bn == 64)
        return 4.1f + L * (0.376f + 0.306f * (rounds - 1)) + 0.8f * tiles / 256.0f;
    return 4.7f + L * (0.367f + 0.485f * (rounds - 1)) + 2.4f * tiles / 256.0f;
}

// tm = 0: a matter for the tiled kernels
Config choose(long long pixels, int taps, int C, int N, bool sums_or_bwd)
{
    Config best = {0, 0, 0, 0, 0};
    float least = tiled_us(pixels, taps * split_over(C, 32), N);
    for(const Cost &o : COSTS) {
        const long long blocks = split_over(pixels, 16 * o.c.tm * o.c.wm) * (long long)split_over(N, 16 * o.c.tn);
        const int steps = taps * split_over(C, 32 * o.c.u);
        if(blocks > 640 || steps < o.c.ks) // (beyond what the numbers were fitted to)
            continue;
        // Those of u = 2 to up to 2e10 operations, which their numbers were fitted to.  Of 120 problems of 1.6e10 to 1e11 ten would take
        // them beyond: nine 2 to 39 % faster (52x16x16 5x5 512->64 54 -> 37 us), one 11 % slower (20x25x25 5x5 384->160 74 -> 82).
        // Passes with sums for norms and backward passes keep the order of sums of u = 1: a step of Adam and norms of few values
        // pass a difference in rounding on.  The loss of a ResNet-50's third step, u = 2 against 1: both ways 5.6 % apart at 19x160x160, 2.8 at
        // 90x144x144, backward alone 5.7 and 2.6; a step at 23x193x193 takes 4060 to 4080 us with and without.  (A forward convolution
        // without a norm behind it takes u = 2 in a training step as well: a call does not know what it is part of.)
        if(o.c.u == 2 && (sums_or_bwd || C % 64 || (double)pixels * N * taps * C > 1e10))
            continue;
        const int rounds = split_over(blocks, 256);
        const float us = o.start + split_over(steps, o.c.ks) * (o.step + o.more * rounds) + o.round * rounds;
        // u = 2 has to be cheaper by more than the numbers are off.  Of 1200 problems of 64 to 2048 channels 24 were 4 to 15 % slower than what
        // u = 2 takes the place of without these lines, 4 with them (the worst 1x49x49 3x3 1536->272 41 -> 47 us); 538 and 515 4 % and more faster.
        // (Layers of a few us lose what little they gained: one image through ResNet-50 328 us without, 333 with them.)
        if(us < least * (o.c.u == 2 && best.u != 2 ? best.tm ? 0.95f : 0.86f : 1.0f)) {
            least = us;
            best = o.c;
        }
    }
    return best;
}

Config config_of(const StreamF16 &g, bool sums)
{
    const int s = g.bwd ? g.stride : 1;
    const long long pixels = (long long)g.batch * ((g.OH + s - 1) / s) * ((g.OW + s - 1) / s) * s * s;
    const int taps = ((g.R + s - 1) / s) * ((g.S + s - 1) / s);
    return choose(pixels, taps, g.C, g.N, sums || g.bwd);
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
        if(c.Tr > 31 || c.Ts > 31)
            return false;
        c.by_OH = div_by(c.OH > 0 ? c.OH : 1);
        c.by_OW = div_by(c.OW > 0 ? c.OW : 1);
        c.by_Ts = div_by(c.Ts ? c.Ts : 1);
        c.M = g.batch * c.OH * c.OW;
    }
    return true;
}

template <bool SUMS, typename A> int launch_as(const A &k, const Config &cf, hipStream_t st)
{
    const int threads = 64 * cf.ks * cf.wm;
#define GO(TM, TN, U, DEPTH, MAXW)                                                                                          \
    do {                                                                                                                    \
        auto kern = stream_f16_k<TM, TN, U, DEPTH, MAXW, SUMS, A>;                                                                  \
        constexpr size_t lds = wave_lds<TM, TN, U, DEPTH>();                                                                    \
        static const hipError_t attr = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize,   \
                                                           MAXW * lds);                                                     \
        if(attr != hipSuccess)                                                                                              \
            return (int)attr;                                                                                               \
        kern<<<k.blocks, threads, lds *(threads / 64), st>>>(k);                                                       \
    } while(0)
    if constexpr(!SUMS && sizeof(A) == sizeof(Args1)) { // (forward, without sums)
        if(cf.u == 2) {
            if(cf.tm == 4 && cf.tn == 4)
                GO(4, 4, 2, 2, 4);
            else if(cf.tm == 4)
                GO(4, 2, 2, 0, 8);
            else if(cf.tm == 2)
                GO(2, 2, 2, 2, 8);
            else
                GO(1, 1, 2, 4, 8);
            SAGA_CHECK_LAUNCH();
            return 0;
        }
    }
    if(cf.tm == 4 && cf.tn == 4)
        GO(4, 4, 1, 3, 4);
    else if(cf.tm == 4)
        GO(4, 2, 1, 3, 8);
    else if(cf.tm == 2)
        GO(2, 2, 1, 4, 8);
    else
        GO(1, 1, 1, 8, 8);
#undef GO
    SAGA_CHECK_LAUNCH();
    return 0;
}

} // namespace

bool stream_f16_wanted(const StreamF16 &g) { return config_of(g, g.sums).tm > 0; }

int stream_f16_sum_rows(const StreamF16 &g)
{
    const Config cf = config_of(g, true);
    const int s = g.bwd ? g.stride : 1;
    const long long M = (long long)g.batch * ((g.OH + s - 1) / s) * ((g.OW + s - 1) / s);
    return cf.tm ? (int)((M + 16 * cf.tm * cf.wm - 1) / (16 * cf.tm * cf.wm)) * s * s : 0;
}

int stream_f16_launch(const StreamF16 &g, hipStream_t st, int *sum_rows)
{
    Args k = {};
    k.g = g;
    const long long out_rows = (long long)g.batch * g.OH * g.OW;
    const long long widest = out_rows * std::max({g.ldo, g.bn_flags & SAGA_BN_ADD ? g.ldz : 0, g.bq_x ? g.bq_ldx : 0}) * 2;
    if(widest >= OOB)
        return SAGA_HIP_EUNSUPPORTED;
    k.g.out_bytes = (unsigned)(out_rows * g.ldo * 2);
    k.g.z_bytes = g.bn_flags & SAGA_BN_ADD ? (unsigned)(out_rows * g.ldz * 2) : 0;
    k.g.bq_bytes = g.bq_x ? (unsigned)(out_rows * g.bq_ldx * 2) : 0;
    if(g.C % 8 || g.lda % 8 || !g.a_bytes || !g.b_bytes || !classes(k))
        return SAGA_HIP_EUNSUPPORTED;
    const Config cf = config_of(g, g.sums);
    if(!cf.tm)
        return SAGA_HIP_EUNSUPPORTED;
    while((1 << k.ks_log2) < cf.ks)
        k.ks_log2++;
    k.WM = cf.wm;
    k.S = (g.C + 32 * cf.u - 1) / (32 * cf.u);
    k.by_S = div_by(k.S);
    k.nblk_q = (g.N + 16 * cf.tn - 1) / (16 * cf.tn);
    k.by_q = div_by(k.nblk_q);
    // the larger operand is the one that each die should fetch once
    k.q_outer = (long long)g.N * g.R * g.S > (long long)g.batch * g.IH * g.IW;
    long long blocks = 0;
    int rows = 0;
    for(int i = 0; i < k.nclasses; i++) {
        k.cls[i].block0 = (int)blocks;
        k.cls[i].row0 = rows;
        k.cls[i].nm = (k.cls[i].M + 16 * cf.tm * cf.wm - 1) / (16 * cf.tm * cf.wm);
        k.cls[i].by_nm = div_by(k.cls[i].nm > 0 ? k.cls[i].nm : 1);
        rows += k.cls[i].nm;
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
