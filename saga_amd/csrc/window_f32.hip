// fp32 convolutions on the bf16 matrix unit (split_f32.hpp), each image position read and split once per slice of channels and
// not once per tap.
//
// A block owns 32*TM*WM output pixels, consecutive in (sample, row, column), and 32*WN output channels; KS groups of WM x WN
// wavefronts share the reduction.  What the pixels see of the input under any tap is consecutive in (sample, position) too:
// the window.  For every slice of 8*KG channels a group loads its window in fours of positions, splits it into three parts,
// eight channels to 16 bytes, and leaves it in LDS, where every tap is an offset; the filter comes packed, in the order of the
// lanes (stream_f32.hip), from the caches to registers.
//
// On small grids a wavefront has a SIMD for itself, so what can be done beside the matrix instructions is: the next slice is
// split and written to the window's other half, one position of a lane's four at a time, between this slice's steps, and
// the loads of the one after follow as registers fall free.  Steps are unrolled and loads are issued unconditionally (behind the
// last slice again), so that the compiler knows how many are on their way behind the one it waits for.
//
// What bounds it (us, launch included, packing not; before: fp32 matrix instructions, tiles in LDS or operands straight from
// memory): 3x3 64->64 at 256x56x56 521 -> 289, 205 TFLOP/s of fp32 work or 1230 of bf16, near what this card's matrix unit keeps up.
// 3x3 256->256 at 8x14x14 28 -> 17, of which the matrix instructions take 5: the launch 3, finding the window and the first
// slice 2, the filter from the L2 (4 KB per 16 channels and 32 pixels x 32 channels) most of the rest.  1x1 256->1024 at 8x14x14 16.5 ->
// 10.6: trips to memory, four slices one behind the other.
// Operands without three parts cost the wavefronts that meet them their share again in fp32 products, loaded without staging: 3x3 64->64 at
// 256x56x56 in 360 us, 320 with one NaN in x and 1030 with nothing else (the kernel for fp32 products 520).
#include "split_f32.hpp"
#include "out_f32.hpp"
#include "window_f32.hpp"

#include <algorithm>

namespace {

struct WinArgs {
    const float *p;
    const void *q;
    unsigned p_bytes, q_bytes;
    int M, C, T, Ts; // pixels, reduction channels, taps, taps of a row
    int IH, IW, iy0, ix0, istep, tstep;
    int plane4, quads, WM, WN, KS, nblk_q, blocks;
    int pool; // 1: M counts the pixels of 2x2 windows, ow and oh the windows
    FastDiv ow, oh, blk;
    long long p_sn, p_sc;
    OutArgs o;
};

constexpr unsigned OOB = OUT_NOWHERE;

__device__ __forceinline__ float4_t load4(__amdgpu_buffer_rsrc_t r, unsigned v, unsigned s)
{
    return __builtin_bit_cast(float4_t, __builtin_amdgcn_raw_buffer_load_b128(r, v, s, 0));
}

// Position v of a window is slot (v % 4) * pitch + v / 4 of 16 bytes: with a pitch of 4 mod 8 writes, four positions apart, and
// reads, one apart from a multiple of four on, fall into different banks (a tap beside begins between two: 35 % of the LDS unit's cycles
// are bank conflicts under nine taps by its counter, 1 % under one).  One of the fours is never written by positions: zeros, for taps outside.
__host__ __device__ constexpr int window_pitch(int quads) { return quads + ((4 - quads) & 7); }
constexpr int window_bytes(int quads, int kg) { return 3 * kg * 4 * window_pitch(quads) * 16; }

// APART: one tap at a stride; the window is the positions of the block's pixels and nothing between them, loaded one by one.
// POOL: a max pooling of 2x2 windows behind it (one group; out_f32.hpp).
template <int TM, int DEPTH, int KG, int NR, int TAPS, bool APART, bool EX, bool POOL>
__global__ void __launch_bounds__(512) stream_f32_k_window(WinArgs g)
{
    extern __shared__ __attribute__((aligned(16))) char lds[];
    __shared__ __attribute__((aligned(16))) float chan[2][EX ? 256 : 1]; // scale and shift of the block's channels
    const int tid = threadIdx.x, lane = tid & 63, fr = lane & 31, fk = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int WN = g.WN, WM = g.WM, GW = WM * WN, KS = g.KS; // powers of two
    int ks = 0, wg = wave, wm = 0; // group, wavefront of the group
    while(wg >= GW) {
        wg -= GW;
        ks++;
    }
    int wn = wg;
    while(wn >= WN) {
        wn -= WN;
        wm++;
    }
    const int b = xcd_remap(blockIdx.x, g.blocks);
    const int bm = g.blk.div(b), bq = b - bm * g.nblk_q;
    const int m0 = bm * (32 * TM * WM), n0 = bq * (32 * WN), nw = n0 + 32 * wn;
    const __amdgpu_buffer_rsrc_t rp = __builtin_amdgcn_make_buffer_rsrc((void *)g.p, 0, (int)g.p_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rq = __builtin_amdgcn_make_buffer_rsrc((void *)g.q, 0, (int)g.q_bytes, 0x00020000);

    // every group goes through as many slices; those that are not there are zeros
    const int S16 = (g.C + 15) / 16, total = (S16 + KG / 2 - 1) / (KG / 2), rounds = (total + KS - 1) / KS, s0 = ks * rounds;
    constexpr int STEPS = TAPS * (KG / 2);
    static_assert(STEPS % DEPTH == 0, "the ring goes round in every slice");
    float4_t qr[DEPTH][3];
    const unsigned qoff = nw < g.o.N ? (unsigned)(nw / 32) * (unsigned)(g.T * S16 * 3072) + lane * 16 : OOB;
    auto load_q = [&](int slice, int k) {
        const int st = slice * (KG / 2) + k % (KG / 2);
        const unsigned off = (unsigned)(k % STEPS / (KG / 2) * S16 + (st < S16 ? st : S16 - 1)) * 3072u; // (the window holds zeros there)
#pragma unroll
        for(int h = 0; h < 3; h++)
            qr[k % DEPTH][h] = load4(rq, qoff + 1024 * h, off);
    };
#pragma unroll
    for(int k = 0; k < DEPTH; k++)
        load_q(s0, k);

    // the window
    const int pitch = window_pitch(g.quads), zero = g.quads - 1, half = 3 * KG * 4 * pitch * 16;
    char *const win = lds + ks * 2 * half;
    const int last = m0 + 32 * TM * WM < g.M ? m0 + 32 * TM * WM - 1 : g.M - 1;
    const int dh = g.tstep * g.IW, dw = g.tstep;
    auto place = [&](int m, int &n, int &oy, int &ox) { place_pixel<POOL>(g.ow, g.oh, m, n, oy, ox); };
    auto virt = [&](int n, int oy, int ox) { return n * g.plane4 + (oy * g.istep + g.iy0) * g.IW + ox * g.istep + g.ix0; };
    int n_a, y_a, x_a, n_z, y_z, x_z;
    place(m0, n_a, y_a, x_a);
    place(last, n_z, y_z, x_z);
    const int reach = (TAPS / g.Ts - 1) * dh + (g.Ts - 1) * dw; // of one sign
    const int v0 = virt(n_a, y_a, x_a) + (reach < 0 ? reach : 0), v1 = virt(n_z, y_z, x_z) + (reach > 0 ? reach : 0);
    const int lo = (v0 > n_a * g.plane4 ? v0 : n_a * g.plane4) & ~3;
    const int end = n_z * g.plane4 + g.IH * g.IW - 1, hi = v1 < end ? v1 : end;
    const int nq = hi >= lo ? ((hi - lo) >> 2) + 1 : 0;
    // this lane's loads: four positions (APART: one) of eight channels in every round
    constexpr int QW = 64 / KG; // fours of positions of a wavefront
    const int kg = lane / QW;
    constexpr int EACH = APART ? 1 : 4;
    unsigned xoff[NR];
    int xslot[NR];
#pragma unroll
    for(int r = 0; r < NR; r++) {
        const int q = (r * GW + wg) * QW + lane % QW, v = lo + 4 * q;
        int n = n_a; // a window sees few samples
        while(v >= (n + 1) * g.plane4 && n < n_z)
            n++;
        const bool in = q < nq;
        xoff[r] = in ? (unsigned)((n * g.p_sn + (v - n * g.plane4) + 8 * kg * g.p_sc) * 4) : OOB;
        xslot[r] = in ? (kg * 4 * pitch + q) * 16 : -1;
        if constexpr(APART) {
            const int m = m0 + q;
            int nn, oy, ox;
            place(m <= last ? m : last, nn, oy, ox);
            const int iy = oy * g.istep + g.iy0, ix = ox * g.istep + g.ix0;
            const bool there = m <= last && (unsigned)iy < (unsigned)g.IH && (unsigned)ix < (unsigned)g.IW;
            xoff[r] = there ? (unsigned)((nn * g.p_sn + iy * g.IW + ix + 8 * kg * g.p_sc) * 4) : OOB;
            xslot[r] = q < 32 * TM * WM ? ((kg * 4 + (q & 3)) * pitch + (q >> 2)) * 16 : -1;
        }
    }
    const unsigned psc4 = (unsigned)(g.p_sc * 4);
    float xr[NR][8][EACH];
    auto load_x = [&](int r, int slice) {
        const unsigned v = slice * 8 * KG + 8 * kg < g.C ? xoff[r] : OOB; // channels come in eights
        const int c0 = (slice < total ? slice : total - 1) * 8 * KG;
#pragma unroll
        for(int j = 0; j < 8; j++)
            if constexpr(APART) {
                xr[r][j][0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rp, v, (unsigned)(c0 + j) * psc4, 0));
            } else {
                const float4_t four = load4(rp, v, (unsigned)(c0 + j) * psc4);
#pragma unroll
                for(int e = 0; e < 4; e++)
                    xr[r][j][e] = four[e];
            }
    };
    auto write_x = [&](int unit, char *to) {
        const int r = unit / EACH, e = unit % EACH;
        float x[8];
#pragma unroll
        for(int j = 0; j < 8; j++)
            x[j] = xr[r][j][e];
        Parts p;
        split3(x, p);
        if(xslot[r] >= 0) {
#pragma unroll
            for(int h = 0; h < 3; h++)
                *(uint4_t *)(to + xslot[r] + (h * KG * 4 + e) * pitch * 16) = p.v[h];
        }
    };
#pragma unroll
    for(int r = 0; r < NR; r++)
        load_x(r, s0);

    EpilogueF32::Raw raw;
    if(EX && g.o.e.affine() && tid < 32 * WN)
        raw = g.o.e.fetch(n0 + tid < g.o.N ? n0 + tid : g.o.N - 1);

    // this lane's pixels: where they are in the window under the first tap, and one bit per tap that falls inside the image
    int at[TM], pn[TM], py[TM], px[TM];
    unsigned mask[TM];
    bool ok[TM];
#pragma unroll
    for(int i = 0; i < TM; i++) {
        const int m = m0 + 32 * (TM * wm + i) + fr;
        ok[i] = m < g.M;
        place(ok[i] ? m : 0, pn[i], py[i], px[i]);
        at[i] = APART ? m - m0 : virt(pn[i], py[i], px[i]) - lo;
        unsigned cols = 0;
        int ix = px[i] * g.istep + g.ix0, iy = py[i] * g.istep + g.iy0;
        for(int e = 0; e < g.Ts; e++, ix += g.tstep)
            cols |= ok[i] && (unsigned)ix < (unsigned)g.IW ? 1u << e : 0u;
        mask[i] = 0;
        for(int a = 0; a < TAPS; a += g.Ts, iy += g.tstep)
            mask[i] |= (unsigned)iy < (unsigned)g.IH ? cols << a : 0u;
    }
    for(int k = lane + 64 * wg; k < 6 * KG; k += 64 * GW)
        *(float4_t *)(win + (k * 4 * pitch + zero) * 16) = float4_t{0, 0, 0, 0};

    float16_t acc[TM], low[TM]; // the products of the leading parts, and all others (split_f32.hpp)
#pragma unroll
    for(int i = 0; i < TM; i++)
#pragma unroll
        for(int v = 0; v < 16; v++)
            acc[i][v] = low[i][v] = 0.0f;

    auto meet = [&]() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
#pragma unroll
    for(int u = 0; u < EACH * NR; u++) {
        write_x(u, win);
        if(u % EACH == EACH - 1)
            load_x(u / EACH, s0 + 1);
    }
    meet();

    Parts pp[2][TM];
    for(int it = 0; it < rounds; it++) {
        const int slice = s0 + it;
        const char *from = win + (it & 1) * half;
        char *to = win + (~it & 1) * half;
        auto read_p = [&](int k) {
            const int tp = k / (KG / 2), ty = tp / g.Ts, d = ty * dh + (tp - ty * g.Ts) * dw;
#pragma unroll
            for(int i = 0; i < TM; i++) {
                const int v = at[i] + d;
                const int slot = (mask[i] >> tp) & 1 ? (v & 3) * pitch + (v >> 2) : zero;
                const char *src = from + ((2 * (k % (KG / 2)) + fk) * 4 * pitch + slot) * 16;
#pragma unroll
                for(int h = 0; h < 3; h++)
                    pp[k & 1][i].v[h] = *(const uint4_t *)(src + h * KG * 4 * pitch * 16);
            }
        };
        read_p(0);
#pragma unroll
        for(int k = 0; k < STEPS; k++) {
            if(k + 1 < STEPS)
                read_p(k + 1);
            // one product of all tiles after the other: an instruction that adds to the one before waits for it
#pragma unroll
            for(int j = 0; j < SPLIT_PRODUCTS; j++)
#pragma unroll
                for(int i = 0; i < TM; i++)
                    mfma_split(j, pp[k & 1][i], qr[k % DEPTH], acc[i], low[i]);
            load_q(k + DEPTH < STEPS ? slice : slice + 1, k + DEPTH);
#pragma unroll
            for(int u = k * EACH * NR / STEPS; u < (k + 1) * EACH * NR / STEPS; u++) {
                write_x(u, to);
                if(u % EACH == EACH - 1)
                    load_x(u / EACH, slice + 2);
            }
            __builtin_amdgcn_sched_barrier(0); // or the loads sink to where they are needed
        }
        meet();
    }

    float bad = 0.0f;
#pragma unroll
    for(int i = 0; i < TM; i++)
#pragma unroll
        for(int v = 0; v < 16; v++) {
            acc[i][v] = (acc[i][v] + low[i][v]) * SPLIT_SUM;
            bad = __builtin_fmaf(acc[i][v], 0.0f, bad);
        }
    if(__builtin_amdgcn_ballot_w64(bad != bad)) {
        // An infinity, a NaN or a number next to the largest among the operands has no three parts: this wavefront's share
        // once more, in fp32 products.
#pragma unroll
        for(int i = 0; i < TM; i++)
#pragma unroll
            for(int v = 0; v < 16; v++)
                acc[i][v] = 0.0f;
        const int first = s0 * (KG / 2), behind = first + rounds * (KG / 2) < S16 ? first + rounds * (KG / 2) : S16;
        for(int st = first; st < behind; st++)
            for(int tp = 0; tp < TAPS; tp++) {
                const int ty = tp / g.Ts, d = ty * dh + (tp - ty * g.Ts) * dw;
                float a[TM][8];
#pragma unroll
                for(int i = 0; i < TM; i++) {
                    const long long at0 = pn[i] * g.p_sn + (py[i] * g.istep + g.iy0) * g.IW + px[i] * g.istep + g.ix0 + d + 8 * fk * g.p_sc;
                    const unsigned v = (mask[i] >> tp) & 1 && st * 16 + 8 * fk < g.C ? (unsigned)(at0 * 4) : OOB;
#pragma unroll
                    for(int j = 0; j < 8; j++)
                        a[i][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rp, v, (unsigned)(st * 16 + j) * psc4, 0));
                }
                float4_t q[3];
#pragma unroll
                for(int h = 0; h < 3; h++)
                    q[h] = load4(rq, qoff + 1024 * h, (unsigned)(tp * S16 + st) * 3072u);
#pragma unroll
                for(int j = 0; j < 8; j++)
#pragma unroll
                    for(int i = 0; i < TM; i++)
                        acc[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(joined(q, j), a[i][j], acc[i], 0, 0, 0);
            }
    }

    // acc[i][v]: this lane's pixel i, channel nw + 8*(v/4) + 4*(lane/32) + v%4
    const FourOut<EX, POOL> out(g.o, fk);
    unsigned opos[TM], zpos[TM];
#pragma unroll
    for(int i = 0; i < TM; i++) {
        opos[i] = out.out_at(ok[i], pn[i], py[i], px[i]);
        zpos[i] = out.z_at(ok[i], pn[i], py[i], px[i]);
    }
    if(EX && g.o.e.affine() && tid < 32 * WN)
        g.o.e.leave(raw, chan[0][tid], chan[1][tid]);
    auto channel = [&](int v) { return nw + 8 * v; };
    auto store = [&](unsigned pos, int n, const Four &val, const Four &was, const Four &res) {
        out.store(pos, n, val, was, res, &chan[0][EX ? n - n0 + 4 * fk : 0], &chan[1][EX ? n - n0 + 4 * fk : 0]);
    };
    constexpr int NV = TM * 16;
    if(POOL || KS == 1) {
        if(EX && g.o.e.affine())
            __syncthreads();
#pragma unroll
        for(int i = 0; i < TM; i++) {
            Four before[4], res[4];
#pragma unroll
            for(int v = 0; v < 4; v++) {
                before[v] = out.before(opos[i], channel(v));
                res[v] = out.residual(zpos[i], channel(v));
            }
#pragma unroll
            for(int v = 0; v < 4; v++)
                store(opos[i], channel(v), {acc[i][4 * v], acc[i][4 * v + 1], acc[i][4 * v + 2], acc[i][4 * v + 3]}, before[v], res[v]);
        }
        return;
    }
    // the groups' sums meet in LDS; each wavefront finishes its share of the fours
    float4_t *const red = (float4_t *)lds;
#pragma unroll
    for(int i = 0; i < TM; i++)
#pragma unroll
        for(int v = 0; v < 4; v++)
            red[(wave * (NV / 4) + i * 4 + v) * 64 + lane] = float4_t{acc[i][4 * v], acc[i][4 * v + 1], acc[i][4 * v + 2], acc[i][4 * v + 3]};
    __syncthreads();
#pragma unroll
    for(int f = 0; f < NV / 4; f++) {
        if((f & (KS - 1)) != ks)
            continue;
        const int i = f / 4, v = f % 4;
        const Four before = out.before(opos[i], channel(v)), res = out.residual(zpos[i], channel(v));
        float4_t sum = {0, 0, 0, 0};
        for(int k = 0; k < KS; k++)
            sum += red[((k * GW + wg) * (NV / 4) + f) * 64 + lane];
        store(opos[i], channel(v), {sum[0], sum[1], sum[2], sum[3]}, before, res);
    }
}

// Pixels of a wavefront in 32s (of channels it has 32), wavefronts of a group along the pixels and the channels, groups along the reduction.
struct Config {
    int tm, wm, wn, ks;
};

constexpr int MAX_LDS = 160 * 1024 - 2048 - 512;

// What a window takes: positions that so many pixels see, in fours, and one four of zeros; 0: the order of the pixels is not
// the order of what they see (a row or an image whose first or last pixel sees nothing of it).
int window_quads(const WinArgs &g, int Tr, int pixels)
{
    if(g.T == 1 && g.istep > 1)
        return (pixels + 3) / 4 + 1;
    const int OW = (int)g.ow.d << g.pool, OH = (int)g.oh.d << g.pool;
    auto sees = [&](int count, int first, int n, int size) {
        const int reach = (n - 1) * g.tstep;
        return (count - 1) * g.istep + first + std::min(reach, 0) < size && first + std::max(reach, 0) >= 0;
    };
    if(!sees(OH, g.iy0, Tr, g.IH) || !sees(OW, g.ix0, g.Ts, g.IW))
        return 0;
    const long long reach = (long long)(Tr - 1) * g.tstep * g.IW + (long long)(g.Ts - 1) * g.tstep;
    if(g.pool) { // windows of two rows and columns; the last one's last pixel is a row below and a column beside its first
        const long long n = pixels / 4 - 1, per = OW / 2, rows = (n + per - 1) / per, images = (n + per * (OH / 2) - 1) / (per * (OH / 2));
        const long long most = 2 * n + rows * std::max(0ll, 2ll * g.IW - OW) + images * std::max(0ll, g.plane4 - (long long)OH * g.IW) + g.IW + 1 +
                               std::llabs(reach) + 1;
        return most <= 1024 ? (int)((most + 3) / 4 + 2) : 0;
    }
    const long long px = pixels - 1, rows = (px + OW - 1) / OW, images = (px + (long long)OW * OH - 1) / ((long long)OW * OH);
    const long long row = (long long)g.istep * (g.IW - OW), image = g.plane4 - (long long)OH * g.istep * g.IW;
    const long long skip = (long long)(g.istep - 1) * g.IW; // rows between those of two rows of pixels
    const long long most = px * g.istep + rows * (std::max(0ll, row) + skip) + images * std::max(0ll, image) + std::llabs(reach) + 1;
    return most <= 1024 ? (int)((most + 3) / 4 + 2) : 0;
}

// The launch of a convolution of `g`; quads 0: none fits.
struct Plan {
    Config cf;
    int quads, nr;
    size_t lds;
};

Plan fit(const WinArgs &g, int Tr, int kg, const Config &cf)
{
    const int waves = cf.wm * cf.wn, at_once = 64 / kg * waves; // fours of positions (apart: positions) loaded in a round
    Plan p = {cf, window_quads(g, Tr, 32 * cf.tm * cf.wm), 0, 0};
    const bool apart = g.T == 1 && g.istep > 1;
    p.nr = ((apart ? 32 * cf.tm * cf.wm : p.quads - 1) + at_once - 1) / at_once;
    p.lds = std::max((size_t)cf.ks * 2 * window_bytes(p.quads, kg), cf.ks > 1 ? (size_t)cf.ks * waves * cf.tm * 4096 : 0);
    if(p.nr > (apart ? 4 : 2) || p.lds > MAX_LDS)
        p.quads = 0;
    return p;
}

// What was measured on small grids (us; tm, wm, wn, ks; launch included, packing not):
//   3x3  64->64   8x56x56  2,2,2,1 15.2  2,2,2,2 15.5  1,2,2,1 16.1  2,1,2,1 16.7   1x1  64->64   8x56x56  1,1,2,1  6.7  2,2,2,1  7.4
//   3x3 128->128  8x28x28  2,1,2,4 15.4  1,1,2,2 16.3  2,1,2,2 16.4  2,1,1,4 20.4   1x1  64->256  8x56x56  2,1,8,1 15.1  2,1,4,1 15.5
//   3x3 256->256  8x14x14  1,1,2,4 17.0  2,1,1,4 17.5  1,1,1,4 17.7  2,1,2,4 23.2   1x1 256->64   8x56x56  1,1,2,1 11.6  2,2,2,1 12.4
//   3x3 512->512  8x7x7    1,1,1,4 21.1  1,1,1,8 21.6  2,1,1,4 26.9  1,1,2,4 28.3   1x1 512->128  8x28x28  1,1,4,2 11.1  1,1,2,2 11.8
//   3x3 128->128 64x28x28  2,4,2,1 77    2,2,4,1 77    2,1,2,1 83    1,1,2,1 93     1x1 1024->256 8x14x14  1,1,2,4 11.5  1,1,1,8 14.3
// 1x1 at stride 2, positions one by one (before: operands straight from memory): 256->512 8x56x56 32 -> 21, 512->1024 8x28x28 36 -> 21,
// 1024->2048 8x14x14 41 -> 27; each lane's four pixels' positions one after the other, with one wavefront of eight at it: 25, 26, 31.
// A wavefront under nine taps has enough to do on 64 pixels as soon as there is one per SIMD or nearly; under one tap, which waits
// for memory, two are better.  Fewer than those: the reduction is split.  Then blocks as large as leave one for three CUs of
// four: those of a group read the same window, and through the L1 the same filter.
Plan tiles_for(const WinArgs &g, int Tr, int kg)
{
    const int taps = g.T, slices = (g.C + 8 * kg - 1) / (8 * kg), columns = (g.o.N + 31) / 32;
    auto tiles = [&](int tm) { return (long long)((g.M + 32 * tm - 1) / (32 * tm)) * columns; };
    // (images of longer rows on small grids: the windows are several times the pixels)
    if(taps > 1 && g.IW > 128 && tiles(2) < 3000)
        return {};
    // 25 taps: four wavefronts next to each other along the pixels share what they load, from 140 blocks of them on; fewer do better
    // with the reduction split (us, the rules below / this: 32->64 at 14x14, 32 images (392 tiles) 10.3 / 12.0, 40 (490) 11.2 / 12.0, 48
    // (588) 13.4 / 12.1, 64 (784) 14.7 / 12.5, 128 (1568) 20.5 / 20.4; 128->192 3x30x30 (510) 23 / 32, 64->96 5x35x35 (576) 19.6 / 18.2,
    // 160->88 20x19x19 (678) 40 / 36, 144->88 174x7x7 (801) 76 / 36; with one column of tiles, 16->32 16x56x56, 14.2 / 15.4)
    if(taps == 25 && g.istep == 1 && columns > 1 && tiles(1) >= 560) {
        const Plan p = fit(g, Tr, kg, {1, 4, 1, 1});
        if(p.quads)
            return p;
    }
    // (25 taps on 64 pixels take more registers than there are; us, 64 / 32: 16->72 82x18x18 backward 60 / 26, 344->16 3x91x91 155 / 81,
    // 96->16 16x96x96 210 / 150, 16->16 75x98x98 179 / 203)
    const long long one = taps == 1 ? 1500 : 750;
    int tm = 1, ks = 1;
    if(taps != 25 && tiles(2) >= one && (g.istep == 1 || taps == 1))
        tm = 2;
    else if(taps > 1 && taps != 25 && tiles(2) >= one / 2 && g.istep == 1)
        tm = 2, ks = 4;
    else
        while(ks < 8 && tiles(1) * ks < (taps == 1 ? 1500 : 800))
            ks *= 2;
    while(ks > 1 && ks > slices)
        ks /= 2;
    for(; tm; tm--)
        for(int k = ks; k; k /= 2) {
            const long long bm = (g.M + 32 * tm - 1) / (32 * tm);
            // (eight wavefronts of one group only where the window is little more than the pixels: such a block fills a CU)
            const int most = taps == 1 || k > 1 || 4 * window_quads(g, Tr, 128) <= 192 ? 8 : 4;
            int wn = 1, wm = 1;
            while(wn < columns && 2 * wn * k <= most && bm * ((columns + 2 * wn - 1) / (2 * wn)) >= 190)
                wn *= 2;
            if(taps > 1 && most == 4 && wn == 4 && bm * ((columns + 1) / 2) >= 2 * 190)
                wn = 2;
            while(taps > 1 && 2 * wm * wn * k <= most && bm * ((columns + wn - 1) / wn) >= 2 * wm * 190)
                wm *= 2;
            for(; wm; wm /= 2) {
                const Plan p = fit(g, Tr, kg, {tm, wm, wn, k});
                if(p.quads)
                    return p;
            }
        }
    return {};
}

// Where operands straight from memory (stream_f32.hip) are faster after all (us, those / windows):
//   1x1 over many pixels and few results, 88->16 247x66x66 95 / 201, 96->24 12x40x40 6.4 / 9.3 (4x40x40 6.2 / 5.3), 256->64 96x56x56
//   111 / 120 (64x56x56 79 / 73), sooner with one slice of channels, 64->64 32x56x56 18 / 22 (24x56x56 17.3 / 16.8); and with a slice
//   of 64 that is not nearly full (window_f32_may), 16->40 217x62x62 48 / 128, 24->144 12x40x40 8.7 / 13.3, 32->192 12x28x28 7.1 / 10.5;
//   blocks of two wavefronts that take a CU's LDS, or under 25 taps: 3x3 at stride 2, 40->64 103x13x13 13 / 21, 472->16 41x13x13
//   30 / 41, 3x3 336->16 1x107x107 36 / 59, 5x5 40->136 3x24x24 19 / 24;
//   few slices over four or eight groups, half of which has one to do less: 3x3 72->152 17x16x16 20 / 30, 72->16 29x37x37 25 / 39;
//   few slices for each of four groups, or one tile, and a last round of blocks that is nearly empty: 3x3 72->128 3x54x54 26 / 32,
//   160->64 2x53x53 22 / 28; of one tile and a large window, over half of the CUs: 104->24 1x70x70 12.5 / 14;
//   one step of channels at stride 2, where a window is four times what its pixels see, and two over many pixels: 3x3 16->296
//   141x48x48 98 / 135, 24->392 61x55x55 122 / 154.
// Of 553 layers under 9 and 25 taps these rules leave 486 to windows, 8 of them (58 without the rules) slower by more than 4 %, one by more than 8.
bool worth(const WinArgs &g, const Plan &p)
{
    const Config &c = p.cf;
    if(g.T == 1)
        return g.o.N > 64 || (g.o.N <= 32 ? g.M < 10000 : (long long)g.M * g.o.N < (g.C <= 64 ? 3ll << 21 : 1ll << 24));
    const int waves = c.wm * c.wn * c.ks, slices = (g.C + 15) / 16;
    const long long blocks = (long long)((g.M + 32 * c.tm * c.wm - 1) / (32 * c.tm * c.wm)) * ((g.o.N + 32 * c.wn - 1) / (32 * c.wn));
    if(g.T == 9 && g.istep > 1 && g.C <= (blocks > 2048 ? 32 : 16))
        return false;
    if(g.T == 9 && (slices + c.ks - 1) / c.ks * c.ks * 2 > slices * 3)
        return false;
    if((160 * 1024) / (p.lds + 2560) > 1)
        return waves > 2 || g.T == 9;
    if(waves <= 2)
        return false;
    if(g.T != 9 || c.ks < 4)
        return true;
    const long long rounds = (blocks + 255) / 256;
    if(rounds > 1 && rounds * 256 * 5 > blocks * 6 && (waves == 4 || slices <= 2 * c.ks))
        return false;
    return !(waves == 4 && g.istep == 1 && p.quads > 30 && blocks > 128);
}

Plan choose(const WinArgs &g, int Tr, int kg)
{
    const Plan p = tiles_for(g, Tr, kg);
    return p.quads && worth(g, p) && !(g.pool && p.cf.ks > 1) ? p : Plan{};
}

bool describe(const WindowConv &c, const SagaTensorView *a, const SagaTensorView *out, bool pool, WinArgs &g)
{
    const int taps = c.Tr * c.Ts, IH = a->dims[2], IW = a->dims[3];
    // A max pooling behind it: windows of two rows see more of the input, the more the longer its rows.  us, packing, convolution and pooling /
    // packing and this: 5x5 32->64 at 64x14x14 22 / 17, at 512x14x14 80 / 67; 3x3 16->32 64x32x32 22 / 14, 64->64 32x56x56 63 / 54, 128->128
    // 16x56x56 98 / 89, 256->256 8x28x28 56 / 52, 512->512 64x14x14 306 / 304; 128->128 3x90x90 56 / 58, 8x112x112 173 / 200.
    if(pool && (taps == 1 || c.istep != 1 || IW > 64))
        return false;
    if(!window_f32_may(c, a->dims[1], IH, IW, out->dims[2] << pool, out->dims[3] << pool) ||
       (IW > 1 && a->strides[3] != 1) || (IH > 1 && a->strides[2] != IW))
        return false;
    const long long pixels = ((long long)out->dims[0] * out->dims[2] * out->dims[3]) << (2 * pool);
    const long long plane4 = ((long long)IH * IW + 3) / 4 * 4;
    if(pixels < 256 || pixels >= 1ll << 30 || (out->dims[0] + 1ll) * plane4 >= 1ll << 30)
        return false;
    g.p = (const float *)a->ptr;
    g.p_bytes = c.a_bytes;
    g.o.N = out->dims[1];
    g.C = a->dims[1];
    g.T = taps;
    g.Ts = c.Ts;
    g.IH = IH;
    g.IW = IW;
    g.iy0 = c.iy0;
    g.ix0 = c.ix0;
    g.istep = c.istep;
    g.tstep = c.tstep;
    g.pool = pool;
    g.M = (int)pixels;
    g.plane4 = (int)plane4;
    g.ow = fast_div(out->dims[3]);
    g.oh = fast_div(out->dims[2]);
    g.p_sn = a->strides[0];
    g.p_sc = a->strides[1];
    return true;
}

int slice_groups(int taps) { return taps == 1 ? 8 : 2; } // eights of channels; under one tap a slice of sixteen waits for memory longer than it works

template <int KG, int TAPS, int DEPTH, bool APART, bool EX, bool POOL = false> int launch_as(const WinArgs &g, const Plan &p, hipStream_t st)
{
#define GO(TM, NR)                                                                                                         \
    do {                                                                                                               \
        auto kern = stream_f32_k_window<TM, DEPTH, KG, NR, TAPS, APART, EX, POOL>;                                                  \
        static const hipError_t attr = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, MAX_LDS); \
        if(attr != hipSuccess)                                                                                         \
            return (int)attr;                                                                                          \
        kern<<<g.blocks, 64 * g.WM * g.WN * g.KS, p.lds, st>>>(g);                                                              \
    } while(0)
    if constexpr(APART)
        if(p.nr > 2) { // (a block of one or two wavefronts)
            if(p.cf.tm == 1)
                GO(1, 4);
            else
                GO(2, 4);
            SAGA_CHECK_LAUNCH();
            return 0;
        }
    if constexpr(TAPS == 25) {
        if(p.nr == 1)
            GO(1, 1);
        else
            GO(1, 2);
    } else if(p.cf.tm == 1 && p.nr == 1)
        GO(1, 1);
    else if(p.cf.tm == 1)
        GO(1, 2);
    else if(p.nr == 1)
        GO(2, 1);
    else
        GO(2, 2);
#undef GO
    SAGA_CHECK_LAUNCH();
    return 0;
}

} // namespace

bool window_f32_may(const WindowConv &c, int channels, int IH, int IW, int OH, int OW)
{
    WinArgs g = {};
    g.T = c.Tr * c.Ts;
    if((g.T != 1 && g.T != 9 && g.T != 25) || channels % 8 || channels < (g.T == 1 ? 48 : 16) || (long long)IH * IW >= 1ll << 30)
        return false;
    g.Ts = c.Ts;
    g.IH = IH;
    g.IW = IW;
    g.iy0 = c.iy0;
    g.ix0 = c.ix0;
    g.istep = c.istep;
    g.tstep = c.tstep;
    g.plane4 = (int)(((long long)IH * IW + 3) / 4 * 4);
    g.ow = fast_div(OW);
    g.oh = fast_div(OH);
    for(int wn = 1; wn <= 8; wn *= 2) // (the smallest tile; with more wavefronts to load its window)
        if(fit(g, c.Tr, slice_groups(g.T), {1, 1, wn, 1}).quads || fit(g, c.Tr, slice_groups(g.T), {1, wn, 1, 1}).quads)
            return true;
    return false;
}

bool window_f32_takes(const WindowConv &c, const SagaTensorView *a, const SagaTensorView *out, bool pool)
{
    WinArgs g = {};
    // (a convolution alone has other kernels for an output out of reach; who asks for a pooling leaves the launches apart then)
    return describe(c, a, out, pool, g) && (!pool || describe_out(out, 1.0f, 0.0f, StreamEpilogue(), g.o)) && choose(g, c.Tr, slice_groups(g.T)).quads;
}

int window_f32_conv(const WindowConv &c, const SagaTensorView *a, const SagaTensorView *out, float alpha, float beta,
                    const StreamEpilogue &e, const void *packed, size_t packed_bytes, bool pool, hipStream_t st)
{
    WinArgs g = {};
    if((pool && (beta != 0.0f || e.z)) || !describe(c, a, out, pool, g) || !describe_out(out, alpha, beta, e, g.o))
        return SAGA_HIP_EUNSUPPORTED;
    const Plan p = choose(g, c.Tr, slice_groups(g.T));
    if(!p.quads)
        return SAGA_HIP_EUNSUPPORTED;
    const long long tile = 32ll * p.cf.tm * p.cf.wm;
    g.q = packed;
    g.q_bytes = (unsigned)packed_bytes;
    g.quads = p.quads;
    g.WM = p.cf.wm;
    g.WN = p.cf.wn;
    g.KS = p.cf.ks;
    g.nblk_q = (g.o.N + 32 * p.cf.wn - 1) / (32 * p.cf.wn);
    g.blk = fast_div(g.nblk_q);
    const long long blocks = (g.M + tile - 1) / tile * g.nblk_q;
    if(blocks >= 1ll << 31)
        return SAGA_HIP_EUNSUPPORTED;
    g.blocks = (int)blocks;
    const bool ex = beta != 0.0f || e.bias || e.bn_s || e.z || e.relu;
    if(g.T == 1) {
        if(g.istep > 1)
            return ex ? launch_as<8, 1, 4, true, true>(g, p, st) : launch_as<8, 1, 4, true, false>(g, p, st);
        return ex ? launch_as<8, 1, 4, false, true>(g, p, st) : launch_as<8, 1, 4, false, false>(g, p, st);
    }
    if(pool)
        return g.T == 9 ? launch_as<2, 9, 3, false, true, true>(g, p, st) : launch_as<2, 25, 5, false, true, true>(g, p, st);
    if(g.T == 9)
        return ex ? launch_as<2, 9, 3, false, true>(g, p, st) : launch_as<2, 9, 3, false, false>(g, p, st);
    return ex ? launch_as<2, 25, 5, false, true>(g, p, st) : launch_as<2, 25, 5, false, false>(g, p, st);
}
