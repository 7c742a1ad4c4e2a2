// fp32 matrix products straight from global memory: on v_mfma_f32_32x32x2_f32, or, from a filter packed for windows
// (window_f32.hip) that are not the faster one after all, on the bf16 matrix unit (split_f32.hpp).
//
// An fp32 matrix instruction keeps the matrix unit busy for 64 cycles with 256 bytes of each operand, so a wavefront
// that loads its own operands from the caches into registers needs 8 - 16 bytes per cycle and SIMD's share of the L1:
// there is nothing for LDS tiles to save, and without them there are no barriers, no LDS traffic and no block-wide
// steps.  A wavefront owns a tile of 32*TM lanes-side elements (pixels of the image written, or columns of the row-major
// GEMM result) x 32*TN others (output channels, or GEMM rows) and a range of the reduction; it loads eight reduction
// indices at a time, DEPTH - 1 steps ahead of the multiplications (the loads of a step are independent, so the compiler's
// counted waits leave the later ones in flight).  The reduction order inside a step is free as long as both operands
// agree: lanes 0 - 31 take indices 0 - 3, lanes 32 - 63 indices 4 - 7, so that an operand whose reduction index is
// contiguous in memory is one 16-byte load.
//
// Small problems fill the chip by splitting the reduction over the KS wavefronts of a block, which add up through LDS
// at the end: one launch, no partial results in memory, a fixed order of additions.
//
// Measured against the LDS-tiled kernels that did all of this before (us; graph replays, launch included): 4096^3 2433 -> 1038 (132 TFLOP/s); 3x3 512->512 at 8x7x7 499 -> 28 with a
// packed filter, 256->256 at 8x14x14 249 -> 27, at 32x14x14 250 -> 79 (94 TFLOP/s); stride-2 backward data of 3x3 128->128
// at 8x56x56 292 -> 45.  A fp32 ResNet-50 batch of 8 7.5 -> 1.5 ms.  What bounds the small ones now is the launch, the first
// trip to memory, and the last round of tiles.
#include "split_f32.hpp"
#include "window_f32.hpp"

#include <string.h>
#include <algorithm>

namespace {

// The lanes-side operand P: PTAP: addressed by tap and channel, the channel count a multiple of eight (also a matrix
// with the lanes' index contiguous); PTAB: by a table of all reduction indices; PROW: reduction index contiguous.
// The other operand Q: QLANE: packed, 1 KB per step of 32 rows in the order of the lanes (stream_pack); QROW: reduction
// index contiguous; QCOL: row index contiguous; QTAB: by the same table; QSPLIT: packed in three parts, 3 KB per step of sixteen.
// (Without windows the parts gain nothing: every tap's operands are split again.  us, QLANE / QSPLIT: 3x3 8->416 at 78x12x12 24 / 37,
// 5x5 8->288 at 243x32x32, stride 2 102 / 161, 7x7 456->40 at 2x15x15 113 / 130, 16->120 at 16x34x34 60 / 52; over 180 such
// layers QSPLIT is 1 to 2 % slower at the median.)
enum { PTAP, PTAB, PROW };
enum { QROW, QCOL, QTAB, QLANE, QSPLIT };

constexpr int MAX_CLASSES = 16;
constexpr int MAX_TABLE = 4096; // reduction indices of a table

// Output pixels whose taps sit at the same distances.  Forward: one class, all pixels.  Backward data at stride s: pixels
// (y, x) with the same y mod s and x mod s; inside a class consecutive taps are a fixed distance apart.
struct Class {
    int oy, ox;   // output pixel = class pixel * ostep + (oy, ox)
    int OH, OW;   // the class's grid
    int r0, s0;   // first tap
    int Tr, Ts;   // taps
    int iy0, ix0; // input position of class pixel (0, 0) under its first tap
    int M;        // class pixels over all samples
    int block0;   // first block
    long long q0; // first byte of the class's rows in a packed filter
};

template <int CLASSES> struct ArgsOf {
    const float *p, *q;
    float *out;
    unsigned p_bytes, q_bytes;
    int N, C; // rows of Q; reduction channels per tap
    int IH, IW, OH, OW;
    int istep, ostep;      // input pixels per class pixel, output pixels per class pixel
    int tstep;             // input pixels per tap (negative: backward)
    int rstep;             // filter rows per tap row
    long long p_sn, p_sc, p_sh, p_sw;
    long long o_sn, o_sc, o_sh, o_sw;
    long long q_sn, q_sc, q_sr, q_ss;
    float alpha, beta;
    EpilogueF32 e;
    int nclasses, nblk_q, blocks, KS;
    Class cls[CLASSES];
};
typedef ArgsOf<MAX_CLASSES> Args;
typedef ArgsOf<1> Args1; // a kilobyte less to fetch before anything else can start

constexpr unsigned OOB = 0x7fffff00u; // beyond every buffer: the load returns zero

__device__ __forceinline__ float load1(__amdgpu_buffer_rsrc_t r, unsigned v, unsigned s)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, v, s, 0));
}
__device__ __forceinline__ float4_t load4(__amdgpu_buffer_rsrc_t r, unsigned v, unsigned s)
{
    return __builtin_bit_cast(float4_t, __builtin_amdgcn_raw_buffer_load_b128(r, v, s, 0));
}

template <int PM, int QM, int TM, int TN, int DEPTH, int MAXW, bool EX, typename A>
__global__ void __launch_bounds__(64 * MAXW) stream_f32_k(A g)
{
    constexpr bool SPLIT = QM == QSPLIT;
    constexpr int HALF = SPLIT ? 8 : 4, STEP = 2 * HALF; // reduction indices per lane and step; of both halves of the lanes
    extern __shared__ __attribute__((aligned(16))) float smem[];
    __shared__ __attribute__((aligned(16))) float chan[2][EX ? 32 * TN : 1]; // scale and shift of the block's channels
    const int tid = threadIdx.x, lane = tid & 63, fr = lane & 31, fk = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int KS = g.KS, WM = (int)(blockDim.x >> 6) / KS;
    const int wm = wave / KS, ks = wave - wm * KS;
    int b = xcd_remap(blockIdx.x, g.blocks), ci = 0;
    while(sizeof(A) > sizeof(Args1) && ci + 1 < g.nclasses && b >= g.cls[ci + 1].block0)
        ci++;
    const Class &c = g.cls[ci];
    b -= c.block0;
    const int bm = b / g.nblk_q, bq = b - bm * g.nblk_q;
    const int m0 = (bm * WM + wm) * (32 * TM), n0 = bq * (32 * TN);
    const int T = c.Tr * c.Ts;
    const __amdgpu_buffer_rsrc_t rp = __builtin_amdgcn_make_buffer_rsrc((void *)g.p, 0, (int)g.p_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rq = __builtin_amdgcn_make_buffer_rsrc((void *)g.q, 0, (int)g.q_bytes, 0x00020000);

    EpilogueF32::Raw raw;
    if(EX && g.e.affine() && tid < 32 * TN)
        raw = g.e.fetch(n0 + tid < g.N ? n0 + tid : g.N - 1);

    // this lane's pixels: byte offset of the first tap (negative outside the image: only valid taps are read) and one
    // bit per tap that falls inside
    int base[TM];
    unsigned long long mask[TM];
    bool ok[TM];
#pragma unroll
    for(int i = 0; i < TM; i++) {
        const int m = m0 + 32 * i + fr;
        ok[i] = m < c.M;
        const int mm = ok[i] ? m : 0;
        const int ox = mm % c.OW, t = mm / c.OW;
        const int oy = t % c.OH, n = t / c.OH;
        const int iy = oy * g.istep + c.iy0, ix = ox * g.istep + c.ix0;
        base[i] = (int)((n * g.p_sn + iy * g.p_sh + ix * g.p_sw + (PM == PTAP ? HALF * fk * g.p_sc : PM == PROW ? HALF * fk : 0)) * 4);
        mask[i] = 0;
        if(PM == PROW || !ok[i])
            mask[i] = ok[i] ? 1 : 0;
        else
            for(int a = 0; a < c.Tr; a++) {
                const int yy = iy + a * g.tstep;
                if(yy < 0 || yy >= g.IH)
                    continue;
                for(int e = 0; e < c.Ts; e++) {
                    const int xx = ix + e * g.tstep;
                    if(xx >= 0 && xx < g.IW)
                        mask[i] |= 1ull << (a * c.Ts + e);
                }
            }
    }
    const int kred = T * g.C;
    unsigned qoff[TN];
    bool nok[TN];
#pragma unroll
    for(int t = 0; t < TN; t++) {
        const int n = n0 + 32 * t + fr;
        nok[t] = n < g.N;
        const long long o = QM == QLANE  ? c.q0 + (long long)(n0 / 32 + t) * (kred / 8) * 1024 + lane * 16
                            : QM == QSPLIT ? c.q0 + (long long)(n0 / 32 + t) * T * ((g.C + 15) / 16) * 3072 + lane * 16
                            : QM == QROW ? ((long long)n * g.q_sn + 4 * fk) * 4
                            : QM == QCOL ? (n + 4 * fk * g.q_sc) * 4
                                         : n * g.q_sn * 4;
        qoff[t] = nok[t] || SPLIT ? (unsigned)o : OOB; // (a packed filter has whole tiles of rows)
    }

    // table: byte offsets of both operands and the tap of every reduction index, eight dead entries behind the last
    int4 *tab = (int4 *)smem;
    const int S8 = PM == PTAB ? (kred + 7) / 8 : SPLIT ? (g.C + 15) / 16 : g.C / 8; // steps per tap; of the whole reduction with a table
    const int total = PM == PTAB ? S8 : S8 * T;
    if constexpr(PM == PTAB) {
        for(int k = tid; k < total * 8 + 8; k += blockDim.x) {
            int4 e = {0, 63, (int)OOB, 0};
            if(k < kred) {
                const int ch = k / T, tap = k - ch * T, a = tap / c.Ts, s = tap - a * c.Ts;
                e.x = (int)((ch * g.p_sc + a * g.tstep * g.p_sh + s * g.tstep * g.p_sw) * 4);
                e.y = tap;
                e.z = (int)((ch * g.q_sc + (c.r0 + a * g.rstep) * g.q_sr + (c.s0 + s * g.rstep) * g.q_ss) * 4);
            }
            tab[k] = e;
        }
        __syncthreads();
    }
    const int s_begin = (int)((long long)ks * total / KS), s_end = (int)((long long)(ks + 1) * total / KS);

    // next step to be loaded: channels 8 * c8 ... of tap (ta, te)
    int s_next = s_begin, tap = PM == PTAB || !total ? 0 : s_begin / S8, c8 = PM == PTAB ? 0 : s_begin - tap * S8;
    int ta = c.Ts ? tap / c.Ts : 0, te = tap - ta * c.Ts;
    unsigned pv[TM];
    const int dh = (int)(g.tstep * g.p_sh * 4), dw = (int)(g.tstep * g.p_sw * 4);
    auto tap_setup = [&]() {
        const int d = PM == PTAP ? ta * dh + te * dw : 0;
#pragma unroll
        for(int i = 0; i < TM; i++)
            pv[i] = (mask[i] >> tap) & 1 ? (unsigned)(base[i] + d) : OOB;
    };
    if(PM != PTAB)
        tap_setup();
    const unsigned psc4 = (unsigned)(g.p_sc * 4), qsc4 = (unsigned)(g.q_sc * 4);

    float pr[DEPTH][TM][HALF];
    float4_t qr[DEPTH][TN][SPLIT ? 3 : 1];
    auto load_step = [&](int u) {
        const bool live = s_next < s_end;
        if constexpr(PM == PTAB) {
            const int4 *e = tab + (live ? s_next : total) * 8 + 4 * fk;
#pragma unroll
            for(int j = 0; j < 4; j++) {
                const int4 w = e[j];
#pragma unroll
                for(int i = 0; i < TM; i++)
                    pr[u][i][j] = load1(rp, (mask[i] >> w.y) & 1 ? (unsigned)(base[i] + w.x) : OOB, 0);
#pragma unroll
                for(int t = 0; t < TN; t++)
                    qr[u][t][0][j] = load1(rq, nok[t] && w.y < 63 ? qoff[t] + (unsigned)w.z : OOB, 0);
            }
        } else {
#pragma unroll
            for(int i = 0; i < TM; i++) {
                const unsigned v = live && (!SPLIT || c8 * 16 + 8 * fk < g.C) ? pv[i] : OOB;
                if constexpr(PM == PROW) {
                    const float4_t f = load4(rp, v, (unsigned)(c8 * 32));
#pragma unroll
                    for(int j = 0; j < 4; j++)
                        pr[u][i][j] = f[j];
                } else {
#pragma unroll
                    for(int j = 0; j < HALF; j++)
                        pr[u][i][j] = load1(rp, v, (unsigned)(c8 * STEP + j) * psc4);
                }
            }
#pragma unroll
            for(int t = 0; t < TN; t++) {
                const unsigned v = live ? qoff[t] : OOB;
                if constexpr(SPLIT) {
#pragma unroll
                    for(int h = 0; h < 3; h++)
                        qr[u][t][h] = load4(rq, v + 1024 * h, (unsigned)(live ? s_next : 0) * 3072u);
                } else if constexpr(QM == QLANE || QM == QROW) {
                    qr[u][t][0] = load4(rq, v, (unsigned)(s_next * (QM == QLANE ? 1024 : 32)));
                } else {
#pragma unroll
                    for(int j = 0; j < 4; j++)
                        qr[u][t][0][j] = load1(rq, v, (unsigned)(s_next * 8 + j) * qsc4);
                }
            }
            if(++c8 == S8) {
                c8 = 0;
                tap++;
                if(++te == c.Ts) {
                    te = 0;
                    ta++;
                }
                if(s_next + 1 < s_end)
                    tap_setup();
            }
        }
        s_next++;
    };

    // split: acc takes the products of the leading parts, low all others (see split3)
    float16_t acc[TM][TN], low[SPLIT ? TM : 1][SPLIT ? TN : 1];
    auto clear = [&]() {
#pragma unroll
        for(int i = 0; i < TM; i++)
#pragma unroll
            for(int t = 0; t < TN; t++)
#pragma unroll
                for(int v = 0; v < 16; v++) {
                    acc[i][t][v] = 0.0f;
                    if constexpr(SPLIT)
                        low[i][t][v] = 0.0f;
                }
    };
    clear();
    auto multiply = [&](const float(&a)[TM][HALF], const float4_t(&b)[TN][SPLIT ? 3 : 1]) {
        if constexpr(SPLIT) {
            Parts p[TM];
#pragma unroll
            for(int i = 0; i < TM; i++)
                split3(a[i], p[i]);
#pragma unroll
            for(int j = 0; j < SPLIT_PRODUCTS; j++) // one product of all tiles after the other: an instruction waits for the one it adds to
#pragma unroll
                for(int i = 0; i < TM; i++)
#pragma unroll
                    for(int t = 0; t < TN; t++)
                        mfma_split(j, p[i], b[t], acc[i][t], low[i][t]);
        } else {
#pragma unroll
            for(int j = 0; j < 4; j++)
#pragma unroll
                for(int i = 0; i < TM; i++)
#pragma unroll
                    for(int t = 0; t < TN; t++)
                        acc[i][t] = __builtin_amdgcn_mfma_f32_32x32x2f32(b[t][0][j], a[i][j], acc[i][t], 0, 0, 0);
        }
    };
    // a matrix whose reduction length is no multiple of eight: the last, partial step, each index tested; requested
    // first, so that a short reduction pays one trip to memory
    float tp[TM][HALF];
    float4_t tq[TN][SPLIT ? 3 : 1];
    const bool tail = !SPLIT && PM != PTAB && g.C % 8 && ks == KS - 1;
    if constexpr(!SPLIT)
    if(tail) {
#pragma unroll
        for(int j = 0; j < 4; j++) {
            const int k = S8 * 8 + 4 * fk + j;
#pragma unroll
            for(int i = 0; i < TM; i++)
                tp[i][j] = load1(rp, ok[i] && k < g.C ? (unsigned)(base[i] + (PM == PROW ? (S8 * 8 + j) * 4 : (int)((S8 * 8 + j) * psc4))) : OOB, 0);
#pragma unroll
            for(int t = 0; t < TN; t++)
                tq[t][0][j] = load1(rq, nok[t] && k < g.C ? qoff[t] + (QM == QROW ? (unsigned)((S8 * 8 + j) * 4) : (unsigned)(S8 * 8 + j) * qsc4) : OOB, 0);
        }
    }
#pragma unroll
    for(int u = 0; u < DEPTH - 1; u++)
        load_step(u);
    for(int s = s_begin; s < s_end; s += DEPTH) {
#pragma unroll
        for(int u = 0; u < DEPTH; u++) {
            load_step((u + DEPTH - 1) % DEPTH);
            if(s + u < s_end)
                multiply(pr[u], qr[u]);
        }
    }
    if constexpr(!SPLIT) {
        if(tail)
            multiply(tp, tq);
    } else {
        float bad = 0.0f;
#pragma unroll
        for(int i = 0; i < TM; i++)
#pragma unroll
            for(int t = 0; t < TN; t++)
#pragma unroll
                for(int v = 0; v < 16; v++) {
                    acc[i][t][v] = (acc[i][t][v] + low[i][t][v]) * SPLIT_SUM;
                    bad = __builtin_fmaf(acc[i][t][v], 0.0f, bad);
                }
        if(__builtin_amdgcn_ballot_w64(bad != bad)) {
            // An infinity, a NaN or a number next to the largest among the operands has no three parts: this wavefront's
            // share once more, in fp32 products.
            clear();
            s_next = s_begin;
            tap = total ? s_begin / S8 : 0;
            c8 = s_begin - tap * S8;
            ta = c.Ts ? tap / c.Ts : 0;
            te = tap - ta * c.Ts;
            tap_setup();
            for(int s = s_begin; s < s_end; s++) {
                load_step(0);
#pragma unroll
                for(int j = 0; j < HALF; j++)
#pragma unroll
                    for(int i = 0; i < TM; i++)
#pragma unroll
                        for(int t = 0; t < TN; t++)
                            acc[i][t] = __builtin_amdgcn_mfma_f32_32x32x2f32(joined(qr[0][t], j), pr[0][i][j], acc[i][t], 0, 0, 0);
            }
        }
    }

    // acc[i][t][v]: pixel m0 + 32*i + lane%32, channel n0 + 32*t + 8*(v/4) + 4*(lane/32) + v%4
    long long opos[TM], zpos[TM];
#pragma unroll
    for(int i = 0; i < TM; i++) {
        const int mm = ok[i] ? m0 + 32 * i + fr : 0;
        const int ox = mm % c.OW, t = mm / c.OW;
        const int oy = t % c.OH, n = t / c.OH;
        const int y = oy * g.ostep + c.oy, x = ox * g.ostep + c.ox;
        opos[i] = n * g.o_sn + y * g.o_sh + x * g.o_sw;
        zpos[i] = n * g.e.z_sn + y * g.e.z_sh + x * g.e.z_sw;
    }
    if(EX && g.e.affine() && tid < 32 * TN)
        g.e.leave(raw, chan[0][tid], chan[1][tid]);
    // what is added to the values is requested for many of them before the first is needed
    auto channel = [&](int t, int v) { return n0 + 32 * t + 8 * (v >> 2) + 4 * fk + (v & 3); };
    auto old = [&](long long op, int t, int v) { const int n = channel(t, v); return g.out[op + (n < g.N ? n : 0) * g.o_sc]; };
    auto residual = [&](long long zp, int t, int v) { const int n = channel(t, v); return g.e.z[zp + (n < g.N ? n : 0) * g.e.z_sc]; };
    auto store = [&](bool pok, long long op, int t, int v, float val, float before, float res) {
        const int n = channel(t, v);
        if(!pok || n >= g.N)
            return;
        val *= g.alpha;
        if constexpr(EX) {
            if(g.beta != 0.0f)
                val += g.beta * before;
            val = g.e.apply(val, chan[0][n - n0], chan[1][n - n0], res);
        }
        g.out[op + n * g.o_sc] = val;
    };
    constexpr int NV = TM * TN * 16;
    if(KS == 1) {
        if(EX && g.e.affine())
            __syncthreads();
#pragma unroll
        for(int i = 0; i < TM; i++)
#pragma unroll
            for(int e0 = 0; e0 < TN * 16; e0 += 8) {
                float before[8] = {}, res[8] = {};
                if(EX && g.beta != 0.0f)
#pragma unroll
                    for(int j = 0; j < 8; j++)
                        before[j] = old(opos[i], (e0 + j) >> 4, (e0 + j) & 15);
                if(EX && g.e.z)
#pragma unroll
                    for(int j = 0; j < 8; j++)
                        res[j] = residual(zpos[i], (e0 + j) >> 4, (e0 + j) & 15);
#pragma unroll
                for(int j = 0; j < 8; j++)
                    store(ok[i], opos[i], (e0 + j) >> 4, (e0 + j) & 15, acc[i][e0 >> 4][(e0 + j) & 15], before[j], res[j]);
            }
        return;
    }
    if(PM == PTAB)
        __syncthreads(); // the table's memory is reused
#pragma unroll
    for(int i = 0; i < TM; i++)
#pragma unroll
        for(int t = 0; t < TN; t++)
#pragma unroll
            for(int v = 0; v < 16; v++)
                smem[(wave * NV + (i * TN + t) * 16 + v) * 64 + lane] = acc[i][t][v];
    const int per = NV / KS; // KS divides 16
    auto place = [&](int j, int &t, int &v) {
        const int e = ks * per + j;
        t = (e >> 4) % TN;
        v = e & 15;
        return TM > 1 && e / (16 * TN);
    };
    auto gather = [&](int j0, float(&before)[4], float(&res)[4]) {
#pragma unroll
        for(int j = 0; j < 4; j++) {
            int t, v;
            const bool hi = place(j0 + (j0 + j < per ? j : 0), t, v);
            if(EX && g.beta != 0.0f)
                before[j] = old(hi ? opos[TM - 1] : opos[0], t, v);
            if(EX && g.e.z)
                res[j] = residual(hi ? zpos[TM - 1] : zpos[0], t, v);
        }
    };
    float before[4] = {}, res[4] = {};
    gather(0, before, res);
    __syncthreads();
    for(int j0 = 0; j0 < per; j0 += 4) {
        if(j0)
            gather(j0, before, res);
#pragma unroll
        for(int j = 0; j < 4; j++) {
            if(j0 + j >= per)
                break;
            int t, v;
            const bool hi = place(j0 + j, t, v);
            float sum = 0.0f;
            for(int k = 0; k < KS; k++)
                sum += smem[((wm * KS + k) * NV + ks * per + j0 + j) * 64 + lane];
            store(hi ? ok[TM - 1] : ok[0], hi ? opos[TM - 1] : opos[0], t, v, sum, before[j], res[j]);
        }
    }
}

// The filter in the order that the kernels' lanes load it: [class][32 rows][step of eight][lane][4], or in three parts [class]
// [32 rows][step of sixteen][part][lane][8].  A 16-byte load whose neighbouring lanes are rows of the filter apart takes the
// address unit four times as long as one of consecutive addresses (73 and 16 cycles for a kilobyte), and that unit, not the
// matrix unit, bounded 32x32 tiles: 3x3 256->256 at 8x14x14 44 -> 34 us, 512->512 at 8x7x7 51 -> 40, this copy included.
constexpr int AS_IT_IS = SAGA_I32; // SagaFilterPackJob::dtype of an fp32 filter that is not split

__device__ __host__ inline long long pack_chunks(const SagaFilterPackJob &g) // of a lane's elements
{
    return (long long)g.T * (g.dtype == AS_IT_IS ? g.C / 8 : (g.C + 15) / 16) * 64 * ((g.N + 31) / 32);
}

__device__ __forceinline__ void pack_chunk(const SagaFilterPackJob &g, long long i)
{
    const int each = g.dtype == AS_IT_IS ? 4 : 8; // elements of a lane
    const int S = (g.C + 2 * each - 1) / (2 * each), steps = g.T * S;
    const int lane = (int)(i & 63);
    const long long q = i >> 6;
    const int tile = (int)(q / steps), step = (int)(q - (long long)tile * steps);
    const int n = tile * 32 + (lane & 31), tap = step / S, ch = (step - tap * S) * 2 * each + each * (lane >> 5);
    const int a = tap / g.Ts, s = tap - a * g.Ts;
    if(g.dtype == SAGA_HALF) { // (window_f16.hip; channels are contiguous)
        half8_t v = {0, 0, 0, 0, 0, 0, 0, 0};
        if(n < g.N && ch < g.C)
            v = *(const half8_t *)((const half_t *)g.w + n * g.w_sn + ch + (g.r0 + a * g.rstep) * g.w_sr + (g.s0 + s * g.rstep) * g.w_ss);
        *((half8_t *)g.packed + i) = v;
        return;
    }
    const float *src = (const float *)g.w + n * g.w_sn + ch * g.w_sc + (g.r0 + a * g.rstep) * g.w_sr + (g.s0 + s * g.rstep) * g.w_ss;
    float v[8] = {};
    if(n < g.N && ch < g.C) { // channels come in eights
#pragma unroll
        for(int j = 0; j < 8; j++)
            if(j < each)
                v[j] = src[j * g.w_sc];
    }
    if(g.dtype == AS_IT_IS) {
        *((float4_t *)g.packed + i) = float4_t{v[0], v[1], v[2], v[3]};
        return;
    }
    Parts p;
    split3_any(v, p);
    float4_t *out = (float4_t *)g.packed + q * 192 + lane;
#pragma unroll
    for(int h = 0; h < 3; h++)
        out[64 * h] = __builtin_bit_cast(float4_t, p.v[h]);
}

constexpr int PACK_CHUNKS = 1024; // per block

__global__ void __launch_bounds__(256) stream_pack(const SagaFilterPackJob *__restrict__ jobs, int njobs)
{
    int lo = 0, hi = njobs - 1;
    while(lo < hi) {
        const int mid = (lo + hi + 1) / 2;
        if(jobs[mid].first_block <= (int)blockIdx.x)
            lo = mid;
        else
            hi = mid - 1;
    }
    const SagaFilterPackJob g = jobs[lo];
    const long long total = pack_chunks(g);
#pragma unroll
    for(int k = 0; k < PACK_CHUNKS / 256; k++) {
        const long long i = (long long)((int)blockIdx.x - g.first_block) * PACK_CHUNKS + k * 256 + threadIdx.x;
        if(i < total)
            pack_chunk(g, i);
    }
}

// one call's filter, the jobs (one per class) as an argument
struct PackArgs {
    int n;
    SagaFilterPackJob job[MAX_CLASSES];
};
__global__ void __launch_bounds__(256) stream_pack_call(PackArgs a)
{
    const SagaFilterPackJob &g = a.job[blockIdx.y];
    const long long total = pack_chunks(g);
    for(long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < total; i += (long long)gridDim.x * 256)
        pack_chunk(g, i);
}

struct Config {
    int tm, tn, ks, wm;
};

// Tile (32*tm x 32*tn per wavefront), wavefronts of a block along the reduction (ks) and along the pixels (wm) for
// `pixels` x N results with `steps` reduction steps of eight.  Splits fill 1024 SIMDs; the limits are where the measured
// times cross (us, tm,tn,ks,wm; launches included).
// Packed filters: the address unit has room, so the smallest tile balances best, four wavefronts to one tile (blocks of
// one tile spread more evenly than blocks of four), unless the reduction is so short that writing the result dominates:
//   3x3   64->64,  8x56x56   1,1,4,1  27.5   1,1,1,4  27.8   2,1,4,1  30.7   1,1,2,2  28.7
//   3x3  256->256, 32x14x14  1,1,4,1  79.1   2,2,4,1  84.3   1,1,2,2  87.9
//   3x3  256->256, 8x14x14   1,1,8,1  26.8   1,1,4,1  28.5   2,1,4,1  32.3
//   3x3  512->512, 8x7x7     1,1,8,1  28.1   1,1,16,1 28.3   1,1,4,1  34.9
//   1x1  256->64,  8x56x56   1,1,1,4  15.6   1,1,2,2  17.1   1,1,4,1  17.9   2,1,1,4  17.6
//   1x1   64->256, 8x56x56   2,2,1,4  18.2   1,1,1,4  20.3
//   3x3   64->64,  32x56x56  1,1,1,4  80.0   2,2,1,4  82.8
// Filters and matrices read in place or through a table: large tiles reuse what they load.
//   1x1 1024->256, 8x14x14   1,1,4,1  18     2,1,4,1  20     1,1,1,4  33
//   1x1 64->256,   8x56x56   2,1,1,4  22     1,1,1,4  23     1,1,4,1  37
Config choose(bool packed, long long pixels, int N, long long steps)
{
    auto tiles = [&](int tm, int tn) { return ((pixels + 32 * tm - 1) / (32 * tm)) * ((N + 32 * tn - 1) / (32 * tn)); };
    const int tn = N > 32 ? 2 : 1;
    const long long t = tiles(1, 1);
    if(packed) {
        if(t >= 3072 && steps <= 32)
            return {2, tn, 1, 4};
        int ks = t < 4096 && steps >= 64 ? 4 : 1;
        while(ks < 16 && t * ks < (steps >= 64 ? 2048 : 1536) && steps >= 16 * ks)
            ks *= 2;
        return {1, 1, ks, ks >= 4 ? 1 : 4 / ks};
    }
    if(tiles(2, tn) >= 2048)
        return {2, tn, 1, 4};
    if(tiles(2, tn) >= 384 && steps >= 128)
        return {2, tn, 4, 1};
    if(tiles(2, 1) >= 256 && steps >= 48)
        return {2, 1, 4, 1};
    if(tiles(2, 1) >= 1536)
        return {2, 1, 1, 4};
    int ks = 1;
    while(ks < 16 && t * ks < 2048 && steps >= 16 * ks)
        ks *= 2;
    return {1, 1, ks, ks >= 4 ? 1 : 4 / ks};
}

template <int PM, int QM, bool EX, typename A> int launch_as(const A &k, const Config &cf, int threads, size_t lds, hipStream_t st)
{
    constexpr int D = QM == QSPLIT ? 2 : 1; // steps are twice as long
#define GO(TM, TN, DEPTH, MAXW)                                                                                        \
    do {                                                                                                               \
        auto kern = stream_f32_k<PM, QM, TM, TN, DEPTH, MAXW, EX, A>;                                                      \
        static const hipError_t attr = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, \
                                                           (MAX_TABLE + 8) * 16);                                      \
        if(attr != hipSuccess)                                                                                         \
            return (int)attr;                                                                                          \
        kern<<<k.blocks, threads, lds, st>>>(k);                                                                       \
    } while(0)
    if(cf.tm == 2 && cf.tn == 2)
        GO(2, 2, D == 2 ? 2 : 3, 4);
    else if(cf.tm == 2)
        GO(2, 1, D == 2 ? 3 : 4, 4);
    else
        GO(1, 1, 6 / D, 16);
#undef GO
    SAGA_CHECK_LAUNCH();
    return 0;
}

template <int PM, int QM> int launch(Args &g, hipStream_t st, long long pixels, long long steps)
{
    const Config cf = choose(QM == QLANE || QM == QSPLIT, pixels, g.N, steps);
    g.KS = cf.ks;
    g.nblk_q = (g.N + 32 * cf.tn - 1) / (32 * cf.tn);
    long long blocks = 0;
    for(int i = 0; i < g.nclasses; i++) {
        g.cls[i].block0 = (int)blocks;
        blocks += ((g.cls[i].M + 32ll * cf.tm * cf.wm - 1) / (32 * cf.tm * cf.wm)) * g.nblk_q;
    }
    if(blocks > 0x7fffffff)
        return SAGA_HIP_EUNSUPPORTED;
    g.blocks = (int)blocks;
    const bool ex = g.beta != 0.0f || g.e.bias || g.e.bn_s || g.e.z || g.e.relu;
    const int threads = 64 * cf.ks * cf.wm;
    size_t lds = cf.ks > 1 ? (size_t)cf.ks * cf.wm * cf.tm * cf.tn * 16 * 256 : 0;
    if(PM == PTAB) {
        int T = 0;
        for(int i = 0; i < g.nclasses; i++)
            T = std::max(T, g.cls[i].Tr * g.cls[i].Ts);
        lds = std::max(lds, (size_t)((T * g.C + 7) / 8 * 8 + 8) * 16);
    }
    if(g.nclasses > 1)
        return ex ? launch_as<PM, QM, true, Args>(g, cf, threads, lds, st) : launch_as<PM, QM, false, Args>(g, cf, threads, lds, st);
    Args1 one;
    memcpy(&one, &g, sizeof(one)); // the same members up to the first class
    return ex ? launch_as<PM, QM, true, Args1>(one, cf, threads, lds, st) : launch_as<PM, QM, false, Args1>(one, cf, threads, lds, st);
}

long long extent(const SagaTensorView *v)
{
    long long e = 1;
    for(int i = 0; i < 4; i++) {
        if(v->strides[i] < 0)
            return -1;
        e += (long long)(v->dims[i] - 1) * v->strides[i];
    }
    return e * 4;
}

int gcd(int a, int b) { return b ? gcd(b, a % b) : a; }

// packed size of a class with that many taps
long long packed_class(bool bwd, const ConvGeom &g, int taps, bool parts)
{
    const int red = bwd ? g.K : g.C, tiles = ((bwd ? g.C : g.K) + 31) / 32;
    return parts ? (long long)taps * ((red + 15) / 16) * tiles * 3072 : (long long)taps * red * tiles * 128;
}

// the classes of a convolution and how its taps step; false if there are too many
bool classes(bool bwd, const ConvGeom &g, Args &a, bool parts = false)
{
    const int s = bwd ? g.stride : 1;
    if(s * s > MAX_CLASSES)
        return false;
    a.nclasses = s * s;
    a.istep = bwd ? 1 : g.stride;
    a.ostep = s;
    const int q = gcd(s, g.dil);
    a.rstep = s / q;
    a.tstep = bwd ? -g.dil / q : g.dil;
    const int OH = bwd ? g.H : g.P, OW = bwd ? g.W : g.Q;
    long long at = 0;
    for(int i = 0; i < a.nclasses; i++) {
        Class &c = a.cls[i];
        c.oy = i / s;
        c.ox = i % s;
        c.OH = (OH - c.oy + s - 1) / s;
        c.OW = (OW - c.ox + s - 1) / s;
        auto axis = [&](int o, int taps, int &first, int &n, int &pos) {
            for(first = 0; first < a.rstep && (o + g.pad - first * g.dil) % s; first++)
                ;
            if(!bwd) {
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
        const long long M = (long long)g.N * c.OH * c.OW;
        if(M >= 1ll << 31)
            return false;
        c.M = (int)M;
        c.q0 = at;
        at += packed_class(bwd, g, c.Tr * c.Ts, parts);
    }
    return true;
}

WindowConv window_of(const Args &k)
{
    const Class &c = k.cls[0];
    return {c.Tr, c.Ts, c.iy0, c.ix0, k.istep, k.tstep, k.p_bytes};
}

// The filter can be read in place (given dense rows, or columns).
bool in_place(bool bwd, const ConvGeom &g) { return g.R == 1 && g.S == 1 && (!bwd || g.stride == 1); }

// What a filter that is packed beforehand is packed for, windows (in three parts) or QLANE.  It is read by calls on images of
// any number and any strides, so that neither counts here.
bool for_windows(bool bwd, const ConvGeom &g, const Args &k)
{
    return k.nclasses == 1 && window_f32_may(window_of(k), bwd ? g.K : g.C, bwd ? g.P : g.H, bwd ? g.Q : g.W, bwd ? g.H : g.P, bwd ? g.W : g.Q);
}

size_t packed_size(bool bwd, const ConvGeom &g, const Args &k, bool parts)
{
    long long n = 0;
    int taps = 0;
    for(int i = 0; i < k.nclasses; i++) {
        n += packed_class(bwd, g, k.cls[i].Tr * k.cls[i].Ts, parts);
        taps = std::max(taps, k.cls[i].Tr * k.cls[i].Ts);
    }
    return taps <= 64 && n <= 0x7ffffe00ll ? (size_t)n : 0;
}

// Windows of a filter that can be read in place: there has to be so much to multiply that the copy does not count (its launch takes
// about 3 us).
bool pays(bool bwd, const ConvGeom &g)
{
    const long long pixels = bwd ? (long long)g.N * g.H * g.W : (long long)g.N * g.P * g.Q;
    return !in_place(bwd, g) || pixels * (bwd ? g.C : g.K) >= 1ll << 24;
}

void describe(bool bwd, const SagaTensorView *w, Args &k)
{
    k.q_sn = bwd ? w->strides[1] : w->strides[0];
    k.q_sc = bwd ? w->strides[0] : w->strides[1];
    k.q_sr = w->strides[2];
    k.q_ss = w->strides[3];
}

static_assert(sizeof(SagaFilterPackJob) == 88, "as it was before it had a dtype");

int pack_jobs(const Args &k, const void *w, char *packed, bool parts, SagaFilterPackJob *jobs)
{
    int n = 0;
    for(int i = 0; i < k.nclasses; i++) {
        const Class &c = k.cls[i];
        if(!c.Tr || !c.Ts)
            continue;
        SagaFilterPackJob &j = jobs[n++];
        j.w = w;
        j.packed = packed + c.q0;
        j.w_sn = k.q_sn; j.w_sc = k.q_sc; j.w_sr = k.q_sr; j.w_ss = k.q_ss;
        j.N = k.N;
        j.C = k.C;
        j.T = c.Tr * c.Ts;
        j.Ts = c.Ts;
        j.r0 = c.r0;
        j.s0 = c.s0;
        j.rstep = k.rstep;
        j.dtype = parts ? SAGA_FLOAT : AS_IT_IS;
        j.first_block = 0;
        j.blocks = stream_pack_blocks(j);
    }
    return n;
}

} // namespace

int stream_pack_blocks(const SagaFilterPackJob &j) { return (int)((pack_chunks(j) + PACK_CHUNKS - 1) / PACK_CHUNKS); }

size_t stream_f32_packed_bytes(bool bwd, const SagaTensorView *a, const SagaTensorView *w, const SagaTensorView *out, const ConvGeom &g)
{
    Args k = {};
    if((bwd ? g.K : g.C) % 8 || g.group != 1 || !classes(bwd, g, k))
        return 0;
    const bool parts = for_windows(bwd, g, k);
    // Windows are not the faster one here, and the filter as it is serves many pixels as well as a packed one (us, that / three parts:
    // 64->352 109x24x24 44 / 58, 48->120 100x40x40 33 / 46; of few pixels, 2048->512 4x7x7, 19.8 / 16.5)
    const long long pixels = (long long)out->dims[0] * out->dims[2] * out->dims[3];
    if(parts && in_place(bwd, g) && w->strides[1] == 1 && pixels >= 4096 && !stream_f32_windows(bwd, a, out, g, true, 0))
        return 0;
    return packed_size(bwd, g, k, parts);
}

int stream_f32_pack_jobs(bool bwd, const SagaTensorView *w, const ConvGeom &g, void *packed, SagaFilterPackJob *jobs)
{
    Args k = {};
    if(!classes(bwd, g, k))
        return 0;
    const bool parts = for_windows(bwd, g, k);
    classes(bwd, g, k, parts);
    k.N = bwd ? g.C : g.K;
    k.C = bwd ? g.K : g.C;
    describe(bwd, w, k);
    return pack_jobs(k, w->ptr, (char *)packed, parts, jobs);
}

int stream_f32_pack(const SagaFilterPackJob *jobs, int njobs, int blocks, hipStream_t st)
{
    stream_pack<<<blocks, 256, 0, st>>>(jobs, njobs);
    SAGA_CHECK_LAUNCH();
    return 0;
}

bool stream_f32_windows(bool bwd, const SagaTensorView *a, const SagaTensorView *out, const ConvGeom &g, bool packed, size_t room, bool pool)
{
    Args k = {};
    const long long bytes = extent(a);
    if(g.group != 1 || (bwd ? g.K : g.C) % 8 || bytes < 0 || bytes > 0x7ffffe00ll || !classes(bwd, g, k) || k.nclasses > 1)
        return false;
    k.p_bytes = (unsigned)bytes;
    const size_t need = packed_size(bwd, g, k, true);
    return need && (packed ? for_windows(bwd, g, k) : pays(bwd, g) && room >= need) && window_f32_takes(window_of(k), a, out, pool);
}

size_t stream_f32_conv_workspace(bool bwd, const SagaTensorView *a, const SagaTensorView *out, const ConvGeom &g)
{
    Args k = {};
    if((bwd ? g.K : g.C) % 8 || g.group != 1 || !classes(bwd, g, k))
        return 0;
    if(stream_f32_windows(bwd, a, out, g, false, ~(size_t)0))
        return packed_size(bwd, g, k, true);
    return in_place(bwd, g) ? 0 : packed_size(bwd, g, k, false);
}

int stream_f32_conv(bool bwd, const SagaTensorView *a, const SagaTensorView *w, const SagaTensorView *out, const ConvGeom &g,
                    float alpha, float beta, const StreamEpilogue &e, const void *packed, void *ws, size_t ws_bytes, hipStream_t st, bool pool)
{
    Args k = {};
    const long long pe = extent(a), qe = extent(w);
    const long long limit = 0x7ffffe00ll;
    // (a pixel outside the image starts at an offset below the tensor; the sum with a valid tap's offset is inside again)
    if(g.group != 1 || pe < 0 || qe < 0 || pe > limit || qe > limit || !classes(bwd, g, k))
        return SAGA_HIP_EUNSUPPORTED;
    k.p = (const float *)a->ptr;
    k.q = (const float *)w->ptr;
    k.out = (float *)out->ptr;
    k.p_bytes = (unsigned)pe;
    k.q_bytes = (unsigned)qe;
    k.N = out->dims[1];
    k.C = a->dims[1];
    k.IH = a->dims[2];
    k.IW = a->dims[3];
    k.p_sn = a->strides[0]; k.p_sc = a->strides[1]; k.p_sh = a->strides[2]; k.p_sw = a->strides[3];
    k.o_sn = out->strides[0]; k.o_sc = out->strides[1]; k.o_sh = out->strides[2]; k.o_sw = out->strides[3];
    describe(bwd, w, k);
    k.alpha = alpha;
    k.beta = beta;
    k.e = epilogue_f32(e);
    const long long pixels = (long long)out->dims[0] * out->dims[2] * out->dims[3];
    const long long steps = ((long long)k.C * g.R * g.S / k.nclasses + 7) / 8;
    int taps = 0;
    for(int i = 0; i < k.nclasses; i++)
        taps = std::max(taps, k.cls[i].Tr * k.cls[i].Ts);
    if(k.C % 8 == 0 && taps <= 64) {
        const size_t room = ws && aligned16(ws) ? ws_bytes : 0;
        // in three parts for windows, or as it is; packed beforehand as for_windows() has it
        auto from = [&](bool parts) {
            const size_t bytes = packed_size(bwd, g, k, parts);
            classes(bwd, g, k, parts);
            if(!packed) {
                PackArgs pa;
                pa.n = pack_jobs(k, w->ptr, (char *)ws, parts, pa.job);
                const dim3 grid(grid_for((long long)bytes / (parts ? 48 : 16) / k.nclasses, 256, 4096), pa.n);
                stream_pack_call<<<grid, 256, 0, st>>>(pa);
            }
            k.q = (const float *)(packed ? packed : ws);
            k.q_bytes = (unsigned)bytes;
            return bytes;
        };
        if(stream_f32_windows(bwd, a, out, g, packed != nullptr, room, pool)) {
            const Args before = k;
            const size_t bytes = from(true);
            const int r = window_f32_conv(window_of(k), a, out, alpha, beta, e, k.q, bytes, pool, st);
            if(pool)
                return r;
            if(r != SAGA_HIP_EUNSUPPORTED || packed)
                return r == SAGA_HIP_EUNSUPPORTED ? launch<PTAP, QSPLIT>(k, st, pixels, steps) : r;
            k = before; // (an output out of its reach)
        }
        if(pool)
            return SAGA_HIP_EUNSUPPORTED;
        if(packed && packed_size(bwd, g, k, for_windows(bwd, g, k))) {
            const bool parts = for_windows(bwd, g, k);
            from(parts);
            return parts ? launch<PTAP, QSPLIT>(k, st, pixels, steps) : launch<PTAP, QLANE>(k, st, pixels, steps);
        }
        const size_t plain = packed_size(bwd, g, k, false);
        // (without room for the copy: through the table, or the kernels that need less)
        if(!in_place(bwd, g) && plain && room >= plain) {
            from(false);
            return launch<PTAP, QLANE>(k, st, pixels, steps);
        }
        // 1x1: the filter as it is, if its rows are dense
        if(in_place(bwd, g) && !bwd && k.q_sc == 1)
            return launch<PTAP, QROW>(k, st, pixels, steps);
        if(in_place(bwd, g) && bwd && k.q_sn == 1)
            return launch<PTAP, QCOL>(k, st, pixels, steps);
    }
    if(!pool && taps <= 63 && (long long)taps * k.C <= MAX_TABLE - 8)
        return launch<PTAB, QTAB>(k, st, pixels, steps);
    return SAGA_HIP_EUNSUPPORTED;
}

int stream_f32_gemm(int tA, int tB, int M, int N, int K, float alpha, const float *A, int lda, const float *B, int ldb,
                    float beta, float *C, int ldc, const float *bias, int relu, hipStream_t st)
{
    Args k = {};
    const long long ae = ((long long)(tA ? K - 1 : M - 1) * lda + (tA ? M : K)) * 4;
    const long long be = ((long long)(tB ? N - 1 : K - 1) * ldb + (tB ? K : N)) * 4;
    if(ae > 0x7ffffe00ll || be > 0x7ffffe00ll)
        return SAGA_HIP_EUNSUPPORTED;
    k.p = B;
    k.q = A;
    k.out = C;
    k.p_bytes = (unsigned)be;
    k.q_bytes = (unsigned)ae;
    k.N = M;
    k.C = K;
    k.IH = k.IW = 1;
    k.istep = k.ostep = 1;
    k.nclasses = 1;
    Class &c = k.cls[0];
    c.OH = 1;
    c.OW = 1; // "sample" n is column n
    c.Tr = c.Ts = 1;
    c.M = N;
    k.p_sn = tB ? ldb : 1;
    k.p_sc = tB ? 1 : ldb;
    k.o_sn = 1;
    k.o_sc = ldc;
    k.q_sn = tA ? 1 : lda;
    k.q_sc = tA ? lda : 1;
    k.alpha = alpha;
    k.beta = beta;
    k.e.relu = relu;
    if(bias) { // per column: read like a residual with no row stride
        k.e.z = bias;
        k.e.z_sn = 1;
    }
    const long long steps = (K + 7) / 8;
    if(tB)
        return tA ? launch<PROW, QCOL>(k, st, N, steps) : launch<PROW, QROW>(k, st, N, steps);
    return tA ? launch<PTAP, QCOL>(k, st, N, steps) : launch<PTAP, QROW>(k, st, N, steps);
}
