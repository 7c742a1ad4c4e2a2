// What the fp16 implicit-GEMM kernels (conv_mfma.hip, window_f16.hip) share: their arguments, and everything they do after
// their main loop.
#pragma once
#include "conv.hpp"

struct GatherArgs {
    const half_t *a;   // gathered operand (x for forward, dy for backward data)
    const half_t *b;   // [Ngemm][taps * Cred]
    half_t *out;       // [M][ldo]
    int M;             // output rows = N * OH * OW
    int Ngemm;         // output channels
    int Cred;          // channels of the gathered tensor (reduction per tap)
    int IH, IW;        // gathered tensor spatial size
    int OH, OW;        // output spatial size
    int R, S;
    int pad, stride, dil;
    int sshift;        // log2(stride), backward data only
    int lda;           // row pitch of the gathered tensor (elements)
    int ldo;           // row pitch of the output
    float alpha, beta;
    int nblk_n;        // number of block columns
    int nblocks;
    unsigned a_bytes;  // extent of the gathered tensor / of b, for range-checked buffer loads
    unsigned b_bytes;
    int classes;       // backward data: stride*stride residue classes of output pixels (1: none)
    int OHc, OWc, Mc;  // pixel grid and row count of one class (Mc = M when classes == 1)
    int blocks_per_class;
    int nactive;       // classes that get blocks
    unsigned char cls_ids[16]; // residue classes that get blocks (classes with no tap are left out)
    // forward only, optional: y = act(conv * sc[c] + sh[c] (+ z)) with sc = s*rsqrt(v+eps),
    // sh = b - m*sc (batch-norm inference folded into the epilogue)
    const float *bn_s, *bn_b, *bn_m, *bn_v;
    float bn_eps;
    int bn_flags;      // SAGA_BN_RELU | SAGA_BN_ADD
    const half_t *z;   // residual, [M][ldz]
    int ldz;
    // backward data only, optional (kernels instantiated with BQ): the output is the gradient of a batch norm's
    // (+ relu) result and this launch is its only writer.  The epilogue masks it with that relu (recomputed from
    // the norm's input as half(fma(x, s*invstd, b - mean*s*invstd)) > 0, what the forward stored), stores the
    // masked gradient and leaves, per block row and channel, sum(g) and sum(g * (x - mean)) in
    // bq_partial[stats_rows][Ngemm][2]: the first pass of the batch norm's backward.
    const half_t *bq_x; // the norm's input, [M][bq_ldx]
    int bq_ldx;
    const float *bq_mean, *bq_s, *bq_invstd, *bq_b;
    int bq_relu;
    float *bq_partial;  // null: no link
    int no_stage;      // the epilogue stores straight from registers (experiment switch SAGA_HIP_NO_STAGED_STORES)
    int b_krsc;        // conv_rows64_wide<.., FLIP>: b is the filter as the forward pass has it (K,R,S,C), not transposed
    // kernels instantiated with SPLIT: the reduction of a tile is shared by ksplit blocks, which leave their fp32 sums in
    // part (see split_reduce)
    int ksplit;
    float4_t *part;
    size_t part_bytes; // room behind part
    unsigned out_bytes; // extent of out, for the epilogue variant that stores through a range-checked buffer (BUFST)
    // optional, alpha == 1: one value per output channel, which the accumulators start from (conv_gather_gemm_dma and
    // stream_f16; bias_done says that the launch took one of them).  Starting from it costs no register and no store path of
    // its own; a pass over the output took 14 - 92 us per up-convolution of a U-Net at 16 x 256x256, 3 % of its step.
    const half_t *bias = nullptr;
    bool bias_done = false;
    const half_t *packed = nullptr; // b in the order of window_f16.hip, where somebody has it
    float *stats;      // forward only, optional: per block row and output channel, sum and sum of
                       // squares of the stored outputs, [ceil(M / BM)][Ngemm][2]
    int stats_rows;    // out: block rows the launch wrote
};

namespace {

typedef __attribute__((address_space(3))) void *lds_ptr_t;

// The MFMA takes the filter tile as its first operand, so a lane ends up with 4 consecutive
// output CHANNELS of one pixel per accumulator group; v_permlane32_swap pairs the two halves
// of the wave and every lane stores (and, for beta != 0, loads) 16 contiguous bytes.

__device__ __forceinline__ unsigned pack2(float a, float b)
{
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    h2 v;
    v[0] = (_Float16)a;
    v[1] = (_Float16)b;
    return __builtin_bit_cast(unsigned, v);
}

// Eight halves at any address of a half; `count` of them are inside the row (the rest reads as zero, and is not written).  Rows of a
// pitch or at an address that is no multiple of 16 bytes take the same accesses of 16 bytes as others (the hardware splits
// them where they cross a line), and smaller ones for the vector in which a row ends.
typedef unsigned any4_t __attribute__((ext_vector_type(4), aligned(2)));
typedef unsigned any1_t __attribute__((aligned(2)));
typedef unsigned vec4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ vec4_t load_any(const half_t *p, int count)
{
    vec4_t o = {0, 0, 0, 0};
    if(count >= 8)
        o = *(const any4_t *)p;
    else
#pragma unroll
        for(int k = 0; k < 4; k++) {
            if(count >= 2 * k + 2)
                o[k] = *(const any1_t *)(p + 2 * k);
            else if(count == 2 * k + 1)
                o[k] = *(const unsigned short *)(p + 2 * k);
        }
    return o;
}
__device__ __forceinline__ void store_any(half_t *p, vec4_t o, int count)
{
    if(count >= 8)
        *(any4_t *)p = o;
    else
#pragma unroll
        for(int k = 0; k < 4; k++) {
            if(count >= 2 * k + 2)
                *(any1_t *)(p + 2 * k) = o[k];
            else if(count == 2 * k + 1)
                *(unsigned short *)(p + 2 * k) = (unsigned short)o[k];
        }
}

// Reads the 32 channels nb .. nb+31 of this lane's pixel row the way the epilogue stores them
// (16 contiguous bytes per lane: the lower half-wave channels 16q .. 16q+7, the upper one
// 16q+8 .. 16q+15) and hands every lane the values of ITS accumulator elements: the same
// half-wave swap as on the way out undoes the regrouping.  All lanes must call it.
// f[v] belongs to channel nb + 8*(v/4) + 4*hi + v%4.  ANY: rows at any address, of any number of channels.
template <bool ANY = false> __device__ __forceinline__ void load_row32(const half_t *row, bool ok, int nb, int ncols, int hi, float (&f)[16])
{
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
#pragma unroll
    for(int q = 0; q < 2; q++) {
        const int n = nb + 16 * q + 8 * hi;
        u4 o = {0, 0, 0, 0};
        if(ok && n < ncols) {
            if constexpr(ANY)
                o = load_any(row + n, ncols - n);
            else
                o = *(const u4 *)(row + n);
        }
        const auto s0 = __builtin_amdgcn_permlane32_swap(o[0], o[2], false, false);
        const auto s1 = __builtin_amdgcn_permlane32_swap(o[1], o[3], false, false);
        const unsigned w[4] = {s0[0], s1[0], s0[1], s1[1]}; // elements 8q .. 8q+7, two per word
#pragma unroll
        for(int e = 0; e < 4; e++) {
            const h2 v = __builtin_bit_cast(h2, w[e]);
            f[8 * q + 2 * e] = (float)v[0];
            f[8 * q + 2 * e + 1] = (float)v[1];
        }
    }
}

// One step of a halving exchange over n live values per lane: the lane with bit M set keeps
// the upper half, its partner the lower half, and each adds what the other held of its half.
// n is a template parameter so that every array index is a constant and the arrays stay in
// registers.  The partner only has to differ in bit M and agree in the bits above it (the bits
// below are exchanged by the later steps), which lets every step run in the vector ALU instead of
// going through the LDS crossbar (ds_bpermute):
//   M = 16: v_permlane16_swap exchanges the odd 16-lane rows of its first operand with the even rows
//           of the second, after which a lane's two results are its own and its partner's value of the
//           half it keeps (the results pass through an opaque statement: hipcc 7.2 otherwise folds the
//           sum of the two results of one swap into twice the first);
//   M = 8, 4: the partner is the mirror lane of the row of 16 / of the half row of 8 (DPP row_mirror,
//           row_half_mirror); M = 2, 1: the lane two / one away inside the quad (DPP quad_perm).
template <int CTRL> __device__ __forceinline__ float dpp_read(float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, false));
}
template <int n, int M, int NV>
__device__ __forceinline__ void halve_exchange(float (&a)[NV], float (&b)[NV], int lane)
{
    static_assert(M == 16 || M == 8 || M == 4 || M == 2 || M == 1, "partner distance");
    if constexpr(M == 16) {
#pragma unroll
        for(int k = 0; k < n / 2; k++) {
            const auto ra = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, a[k]),
                                                             __builtin_bit_cast(unsigned, a[k + n / 2]), false, false);
            const auto rb = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, b[k]),
                                                             __builtin_bit_cast(unsigned, b[k + n / 2]), false, false);
            unsigned a0 = ra[0], a1 = ra[1], b0 = rb[0], b1 = rb[1];
            asm volatile("" : "+v"(a0), "+v"(a1), "+v"(b0), "+v"(b1));
            a[k] = __builtin_bit_cast(float, a0) + __builtin_bit_cast(float, a1);
            b[k] = __builtin_bit_cast(float, b0) + __builtin_bit_cast(float, b1);
        }
    } else {
        constexpr int CTRL = M == 8 ? 0x140 : M == 4 ? 0x141 : M == 2 ? 0x4e : 0xb1;
        const bool up = lane & M;
#pragma unroll
        for(int k = 0; k < n / 2; k++) {
            const float ka = up ? a[k + n / 2] : a[k], sa = up ? a[k] : a[k + n / 2];
            const float kb = up ? b[k + n / 2] : b[k], sb = up ? b[k] : b[k + n / 2];
            a[k] = ka + dpp_read<CTRL>(sa);
            b[k] = kb + dpp_read<CTRL>(sb);
        }
    }
}

// Everything the gather kernels do after their main loop: alpha / beta, the optional batch-norm
// inference fold (+ residual + relu), the 16-byte channel-vector stores and the optional per-channel
// statistics of the stored values.  acc[i][j][v] belongs to row wm + 32*i + lane%32 of the block tile
// and channel n0 + wn + 32*j + 8*(v/4) + 4*(lane/32) + v%4; rowpix(r, ok, pix) names the output pixel of
// row r of the block tile (ok false: nothing is stored).
// Where the output takes 16-byte vectors the values go out through LDS: a wavefront lays its 64x64 tile down
// row by row (128 bytes per row, 16-byte chunks XORed with the row number against bank conflicts) and reads
// it back with eight lanes per row, so that one store instruction writes eight whole 128-byte rows instead of
// 32-byte pieces of 32 rows.  Measured on MI355X at batch 256 (forward): 64 -> 256 channels over 56x56 pixels
// 135 -> 109 us with fully coalesced stores, 128 -> 512 over 28x28 86 -> 74 us.  MASK: rows that are not ok may hold
// non-zero accumulators and have to be kept out of the statistics.  smem: the block's LDS, free for
// reuse once every wavefront has left the main loop (the barriers inside see to that).
// whether gather_epilogue stores through LDS (the producer wavefronts of a block count its barriers)
// (not the 64-channel tiles: their rows are 128 bytes to begin with and the detour measured 3 - 7 % slower)
// Per-channel sum and sum of squares of a wavefront's outputs (as stored, i.e. rounded to fp16), for a batch
// normalisation that follows.  Columns past Ngemm hold zeros in the accumulators and add nothing; so do rows that
// are not ok unless MASK says they may hold anything, in which case they are left out here.  Lanes of one
// half-wave hold different pixels of the same channels: a halving exchange (each step swaps half of the values
// with the lane 16, 8, .. 1 away) leaves every lane - every even lane for 32-channel tiles - with the totals of
// one channel, stats_channel() of the wave tile.
template <int TM, int TN, bool MASK>
__device__ __forceinline__ void stats_lane_totals(float alpha, float16_t (&acc)[TM][TN], const bool (&okr)[TM], int lane,
                                                  float &s_out, float &q_out)
{
    constexpr int NV = TN * 16;
    static_assert(NV == 16 || NV == 32, "stats layout");
    float sv[NV], qv[NV];
#pragma unroll
    for(int j = 0; j < TN; j++)
#pragma unroll
        for(int v = 0; v < 16; v++) {
            float a = 0.0f, q = 0.0f;
            if constexpr(TM == 2) {
                // the two rows of a channel rounded to fp16 as they are stored, in one packed register;
                // sum and sum of squares are one two-element dot product each (fp32 result)
                typedef _Float16 h2 __attribute__((ext_vector_type(2)));
                h2 pr;
                pr[0] = (!MASK || okr[0]) ? (_Float16)(alpha * acc[0][j][v]) : (_Float16)0;
                pr[1] = (!MASK || okr[1]) ? (_Float16)(alpha * acc[1][j][v]) : (_Float16)0;
                const h2 ones = {(_Float16)1, (_Float16)1};
                a = __builtin_amdgcn_fdot2(pr, ones, 0.0f, false);
                q = __builtin_amdgcn_fdot2(pr, pr, 0.0f, false);
            } else {
#pragma unroll
                for(int i = 0; i < TM; i++) {
                    const float r = (!MASK || okr[i]) ? (float)(half_t)(alpha * acc[i][j][v]) : 0.0f;
                    a += r;
                    q += r * r;
                }
            }
            sv[j * 16 + v] = a;
            qv[j * 16 + v] = q;
        }
    if constexpr(NV == 32) {
        halve_exchange<32, 16>(sv, qv, lane);
        halve_exchange<16, 8>(sv, qv, lane);
        halve_exchange<8, 4>(sv, qv, lane);
        halve_exchange<4, 2>(sv, qv, lane);
        halve_exchange<2, 1>(sv, qv, lane);
    } else {
        halve_exchange<16, 16>(sv, qv, lane);
        halve_exchange<8, 8>(sv, qv, lane);
        halve_exchange<4, 4>(sv, qv, lane);
        halve_exchange<2, 2>(sv, qv, lane);
        sv[0] += dpp_read<0xb1>(sv[0]);
        qv[0] += dpp_read<0xb1>(qv[0]);
    }
    s_out = sv[0];
    q_out = qv[0];
}

// The wavefronts stacked along M are added through LDS (red: WGM * BN pairs) in a fixed order and the block's
// [channel][2] row goes to g.stats[stats_row].  The caller has made sure that nobody still reads what red overlays.
template <int TN, int WGM, int WGN, int BN>
__device__ __forceinline__ void stats_block_write(const GatherArgs &g, char *red_mem, int tid, int lane, int wave, int wn,
                                                  int n0, int stats_row, float s0, float q0)
{
    constexpr int NV = TN * 16;
    const int hi = lane >> 5;
    const int idx = NV == 32 ? (lane & 31) : (lane & 31) >> 1;
    const int chl = 32 * (idx >> 4) + 8 * ((idx & 15) >> 2) + 4 * hi + (idx & 3); // channel inside the wave tile
    typedef float float2_t __attribute__((ext_vector_type(2)));
    float2_t *red = (float2_t *)red_mem;
    if(NV == 32 || (lane & 1) == 0) {
        float2_t v2 = {s0, q0};
        red[(wave / WGN) * BN + wn + chl] = v2;
    }
    __syncthreads();
    if(tid < BN && n0 + tid < g.Ngemm) {
        float2_t t = red[tid];
#pragma unroll
        for(int wy = 1; wy < WGM; wy++)
            t += red[wy * BN + tid];
        *(float2_t *)(g.stats + ((int64_t)stats_row * g.Ngemm + n0 + tid) * 2) = t;
    }
}

template <int TM, int TN, int BN, bool BWD> __device__ __forceinline__ bool stores_staged(const GatherArgs &g)
{
    return TM % 2 == 0 && TN == 2 && BN >= 128 && !(BWD && g.classes > 1) && !g.no_stage;
}

// Inference with a folded batch norm: scale = s/sqrt(v+eps) and shift = b - m*scale of the block's BN channels
// as a table in LDS (bnp: 2 * BN floats).  The caller puts barriers around it.
template <int BN> __device__ __forceinline__ void bnfold_table(const GatherArgs &g, float *bnp, int tid, int n0)
{
    if(tid < BN) {
        const int n = n0 + tid;
        float sc = 0.0f, sh = 0.0f;
        if(n < g.Ngemm) {
            sc = g.bn_s[n] * rsqrtf(g.bn_v[n] + g.bn_eps);
            sh = g.bn_b[n] - g.bn_m[n] * sc;
        }
        bnp[tid] = sc;
        bnp[BN + tid] = sh;
    }
}

// BUFST: the direct 16-byte stores go through a range-checked buffer with an out-of-range offset for the lanes that
// have nothing to store, so that every wavefront issues the same number of store instructions whatever its rows
// (a caller that counts outstanding memory operations needs that).
// ROWS: pixel numbers are not those of the rows of the tile.
template <int TM, int TN, int WGM, int WGN, int BN, bool BWD, bool MASK, bool BUFST = false, bool ROWS = false, typename RowPix>
__device__ __forceinline__ void gather_epilogue(const GatherArgs &g, float16_t (&acc)[TM][TN], char *smem, int tid, int lane,
                                                int wave, int wm, int wn, int n0, int stats_row, RowPix rowpix)
{
    // (the table sits behind the tiles that the wavefronts stage their outputs in; the stage memory is free
    // after the last slice)
    float *bnp = (float *)(smem + WGM * WGN * TM * 32 * TN * 64);
    if constexpr(!BWD) {
        if(g.bn_s) {
            __syncthreads(); // every wavefront is done reading the last slice
            bnfold_table<BN>(g, bnp, tid, n0);
            __syncthreads();
        }
    }
    // acc[i][j][v]: pixel wm + 32*i + lane%32, channel wn + 32*j + 8*(v/4) + 4*(lane/32) + v%4
    const int hi = lane >> 5;
    bool okr[TM];
    const bool vec_ok = (g.ldo & 7) == 0 && (g.Ngemm & 7) == 0 && ((uintptr_t)g.out & 15) == 0;
    // through LDS (see above): this wavefront's 64 rows of 128 bytes
    constexpr bool CAN_STAGE = TM % 2 == 0 && TN == 2 && BN >= 128;
    const bool staged = stores_staged<TM, TN, BN, BWD>(g);
    char *stg = smem + wave * (TM * 32 * TN * 64);
    if(staged && !(!BWD && g.bn_s)) // (the fold's barriers have already seen to it)
        __syncthreads();           // every wavefront is done reading the last slice, which the tiles overwrite
    // ANY: rows off the grid of 16 bytes, or ending inside it.  us, one channel at a time, which stood here before / this: 48->398
    // channels, 1x1, 37x25x25 38.9 / 9.6, 16->180, 3x3, 118x29x29 59.0 / 23.7 (400 and 184 channels: 8.8, 23.0).
    auto store = [&](auto any) {
        constexpr bool ANY = decltype(any)::value;
#pragma unroll
        for(int i = 0; i < TM; i++) {
            bool ok;
            int64_t pix;
            rowpix(wm + i * 32 + (lane & 31), ok, pix);
            okr[i] = ok;
            half_t *orow = g.out + pix * g.ldo;
#pragma unroll
            for(int j = 0; j < TN; j++) {
                const int nb = n0 + wn + j * 32;
                float f[16];
#pragma unroll
                for(int v = 0; v < 16; v++)
                    f[v] = g.alpha * acc[i][j][v];
                typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
                if(g.beta != 0.0f) {
                    float old[16];
                    load_row32<ANY>(orow, ok, nb, g.Ngemm, hi, old);
#pragma unroll
                    for(int v = 0; v < 16; v++)
                        f[v] += g.beta * old[v];
                }
                if constexpr(!BWD) {
                    if(g.bn_s) {
                        float zz[16];
                        if(g.bn_flags & SAGA_BN_ADD)
                            load_row32<ANY>(g.z + pix * g.ldz, ok, nb, g.Ngemm, hi, zz);
#pragma unroll
                        for(int q = 0; q < 4; q++) {
                            // scale and shift of the block's channels were put into LDS after the main loop
                            const int cl = wn + j * 32 + 8 * q + 4 * hi;
                            const float4_t sc = *(const float4_t *)(bnp + cl), sh = *(const float4_t *)(bnp + BN + cl);
#pragma unroll
                            for(int e = 0; e < 4; e++) {
                                float t = __builtin_fmaf(f[4 * q + e], sc[e], sh[e]);
                                if(g.bn_flags & SAGA_BN_ADD)
                                    t += zz[4 * q + e];
                                if(g.bn_flags & SAGA_BN_RELU)
                                    t = (t != t) ? t : fmaxf(t, 0.0f);
                                f[4 * q + e] = t;
                            }
                        }
                    }
                }
                // after the swaps: lower half-wave holds channels 0..7 (then 16..23) of the tile,
                // upper half-wave 8..15 (24..31): one store covers 32 contiguous bytes per pixel
                if constexpr(ANY)
                    __builtin_amdgcn_sched_barrier(0); // (one after the other: the registers are the other branch's)
#pragma unroll
                for(int q = 0; q < 2; q++) {
                    const unsigned x0 = pack2(f[8 * q + 0], f[8 * q + 1]), x1 = pack2(f[8 * q + 2], f[8 * q + 3]);
                    const unsigned y0 = pack2(f[8 * q + 4], f[8 * q + 5]), y1 = pack2(f[8 * q + 6], f[8 * q + 7]);
                    const auto s0_ = __builtin_amdgcn_permlane32_swap(x0, y0, false, false);
                    const auto s1_ = __builtin_amdgcn_permlane32_swap(x1, y1, false, false);
                    const int n = nb + 16 * q + 8 * hi;
                    typedef unsigned u4 __attribute__((ext_vector_type(4)));
                    const u4 o = {s0_[0], s1_[0], s0_[1], s1_[1]};
                    if constexpr(BUFST) {
                        const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc((void *)g.out, 0, g.out_bytes, 0x00020000);
                        const unsigned off = (ok && n < g.Ngemm) ? (unsigned)((pix * g.ldo + n) * 2) : 0x7fffff00u;
                        __builtin_amdgcn_raw_buffer_store_b128(o, ro, off, 0, 0);
                    } else if(staged) {
                        const int row = i * 32 + (lane & 31), chunk = 4 * j + 2 * q + hi;
                        *(u4 *)(stg + row * (TN * 64) + ((chunk ^ (row & 7)) << 4)) = o;
                    } else if(ok && n < g.Ngemm) {
                        if constexpr(ANY)
                            store_any(orow + n, o, g.Ngemm - n);
                        else
                            *(u4 *)(orow + n) = o;
                    }
                }
            }
        }
        if constexpr(CAN_STAGE) {
            if(staged) {
                // LDS operations of one wavefront complete in order: its reads below see its writes above
                typedef unsigned u4 __attribute__((ext_vector_type(4)));
                constexpr int CH = TN * 4, RPI_ = 64 / CH; // 16-byte chunks per row, rows per store instruction
                const int chunk = lane % CH;
                const int n = n0 + wn + chunk * 8;
                // (no residue classes here: the pixel number is the row number, and rows * pitch fits 31 bits)
                bool ok0;
                int64_t pix0;
                rowpix(wm + lane / CH, ok0, pix0);
                const int p0 = (int)pix0;
                const int sw = (chunk ^ ((lane / CH) & 7)) << 4; // RPI_ is a multiple of 8: the same for every row of the lane
                static_assert(RPI_ % 8 == 0, "swizzle period");
#pragma unroll
                for(int it = 0; it < TM * 32 / RPI_; it++) {
                    const int row = it * RPI_ + lane / CH;
                    const int p = p0 + it * RPI_;
                    const u4 o = *(const u4 *)(stg + row * (TN * 64) + sw);
                    if constexpr(ROWS) {
                        bool ok;
                        int64_t pix;
                        rowpix(wm + row, ok, pix);
                        if(ok && n < g.Ngemm) {
                            if constexpr(ANY)
                                store_any(g.out + (pix * g.ldo + n), o, g.Ngemm - n);
                            else
                                *(u4 *)(g.out + (pix * g.ldo + n)) = o;
                        }
                    } else if(p < g.M && n < g.Ngemm) {
                        if constexpr(ANY)
                            store_any(g.out + ((int64_t)p * g.ldo + n), o, g.Ngemm - n);
                        else
                            *(u4 *)(g.out + (p * g.ldo + n)) = o;
                    }
                }
            }
        }
    };
    if(BUFST || vec_ok) // (BUFST's callers have made sure)
        store(std::false_type());
    else
        store(std::true_type());
    // Optional: per-channel sum and sum of squares of this block's outputs, for a batch normalisation that follows
    // (stats_lane_totals, stats_block_write).
    if constexpr(!BWD) {
        if(g.stats) {
            float s0, q0;
            stats_lane_totals<TM, TN, MASK>(g.alpha, acc, okr, lane, s0, q0);
            __syncthreads(); // every wavefront is done reading the last slice (and the folded norm's table)
            stats_block_write<TN, WGM, WGN, BN>(g, smem + WGM * WGN * TM * 32 * TN * 64, tid, lane, wave, wn, n0, stats_row,
                                                s0, q0);
        }
    }
}

// The epilogue of a backward-data launch linked to a batch norm's backward (GatherArgs::bq_*): alpha / beta,
// the norm's relu mask, the 16-byte channel-vector stores of the masked gradient and, per channel, the sums
// of that gradient and of gradient * (x - mean) over the block's rows.  Arguments as in gather_epilogue; the
// output must allow the vector stores.
// Registers decide how many blocks a CU holds, so the work is laid out to need few of them: first every
// accumulator is turned into the fp16 value an unlinked launch would store (two per register, half the
// accumulators' footprint); then the wave tile is walked one 32x32 sub-tile at a time, rows inside
// 32-channel columns, eight elements at a time, and the running sums are kept after the first step of the
// halving exchange (8 per lane and sum instead of 16).  okr / pixr: validity and pixel index of this lane's row
// in row block i (rows * pitch of either tensor fits 31 bits, checked on the host); xraw: bnbwd_prefetch's;
// bnp: bnbwd_table's.
typedef unsigned uint4_t __attribute__((ext_vector_type(4)));

// Mean, and the forward's scale and shift for the relu recompute, of the block's BN channels: written to LDS
// (behind the stage memory) by the first BN threads before the main loop, whose barriers publish it.
template <int BN> __device__ __forceinline__ void bnbwd_table(const GatherArgs &g, float *bnp, int tid, int n0)
{
    if(tid < BN) {
        const int n = n0 + tid;
        float mean = 0.0f, sc = 0.0f, sh = 0.0f;
        if(n < g.Ngemm) {
            mean = g.bq_mean[n];
            if(g.bq_relu) {
                sc = g.bq_s[n] * g.bq_invstd[n];
                sh = __builtin_fmaf(-mean, sc, g.bq_b[n]); // the forward's own expression
            }
        }
        bnp[tid] = mean;
        bnp[BN + tid] = sc;
        bnp[2 * BN + tid] = sh;
    }
}

// The norm's input for the linked epilogue below, fetched by the wavefront before its main loop so that the
// data is in registers when the epilogue starts (four dependent trips to memory per block otherwise, which
// nothing hides once every block of a CU reaches its epilogue at the same time): sub-tile t = j*TM + i
// (row block i, 32-channel column j), two 16-byte vectors each, as the stores of the epilogue are laid out.
template <int TM, int TN, int T0, int T1>
__device__ __forceinline__ void bnbwd_prefetch(const GatherArgs &g, int lane, int wn, int n0, const bool (&okr)[TM],
                                               const int (&pixr)[TM], uint4_t (&xraw)[TM * TN][2])
{
    const int hi = lane >> 5;
#pragma unroll
    for(int t = T0; t < T1; t++) {
        const int j = t / TM, i = t % TM;
        const half_t *row = g.bq_x + pixr[i] * g.bq_ldx;
#pragma unroll
        for(int q = 0; q < 2; q++) {
            const int n = n0 + wn + j * 32 + 16 * q + 8 * hi;
            const uint4_t z = {0, 0, 0, 0};
            xraw[t][q] = z;
            if(okr[i] && n < g.Ngemm)
                xraw[t][q] = *(const uint4_t *)(row + n);
        }
    }
}

template <int TM, int TN, int WGM, int WGN, int BN>
__device__ __forceinline__ void gather_epilogue_bnbwd(const GatherArgs &g, float16_t (&acc)[TM][TN], char *smem, int tid,
                                                      int lane, int wave, int wm, int wn, int n0, int stats_row,
                                                      const bool (&okr)[TM], const int (&pixr)[TM],
                                                      uint4_t (&xraw)[TM * TN][2], const float *bnp)
{
    typedef uint4_t u4;
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    const int hi = lane >> 5;
    // phase 1: pk[i][j][4q .. 4q+3] = channels 8q .. 8q+7 of this lane's accumulator elements, as stored
    unsigned pk[TM][TN][8];
#pragma unroll
    for(int j = 0; j < TN; j++)
#pragma unroll
        for(int i = 0; i < TM; i++) {
            float f[16];
#pragma unroll
            for(int v = 0; v < 16; v++)
                f[v] = g.alpha * acc[i][j][v];
            if(g.beta != 0.0f) {
                float old[16];
                load_row32(g.out + pixr[i] * g.ldo, okr[i], n0 + wn + j * 32, g.Ngemm, hi, old);
#pragma unroll
                for(int v = 0; v < 16; v++)
                    f[v] += g.beta * old[v];
            }
#pragma unroll
            for(int e = 0; e < 8; e++) {
                pk[i][j][e] = pack2(f[2 * e], f[2 * e + 1]);
                asm volatile("" : "+v"(pk[i][j][e])); // converted here and now: the accumulator is dead from here on
            }
        }
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads(); // the parameter table is complete (a block may have had no main-loop barrier to publish it)
    // phase 2
    float sres[TN], qres[TN];
    float sv[8], qv[8];
#pragma unroll
    for(int t = 0; t < TM * TN; t++) {
        const int j = t / TM, i = t % TM;
        const int nb = n0 + wn + j * 32;
        const bool ok = okr[i];
        const u4 (&cur)[2] = xraw[t];
        if(i == 0) {
#pragma unroll
            for(int v = 0; v < 8; v++)
                sv[v] = qv[v] = 0.0f;
        }
        // the norm's input in accumulator order (the same half-wave swap as on the way out, undone):
        // wx[c][2*(e/2) .. ] holds elements 8c + 2*ee, 8c + 2*ee + 1 in word ee
        unsigned wx[2][4];
#pragma unroll
        for(int c = 0; c < 2; c++) {
            const auto s0 = __builtin_amdgcn_permlane32_swap(cur[c][0], cur[c][2], false, false);
            const auto s1 = __builtin_amdgcn_permlane32_swap(cur[c][1], cur[c][3], false, false);
            wx[c][0] = s0[0]; wx[c][1] = s1[0]; wx[c][2] = s0[1]; wx[c][3] = s1[1];
        }
        // Elements are handled eight at a time: the four of channel group q = half and the four of group
        // q + 2, which are the partners of the first step of the halving exchange (element k with k + 8; the
        // lane with bit 16 set keeps the upper one, its partner 16 lanes away the lower one) - that step is
        // folded into the running sums right away, so only eight gradients and products are live at a time.
#pragma unroll
        for(int half = 0; half < 2; half++) {
            float gf[2][4], gq[2][4];
#pragma unroll
            for(int side = 0; side < 2; side++) {
                const int q = half + 2 * side;
                // the table is read again for every sub-tile (the opaque index keeps the compiler from holding
                // a column's 48 parameters in registers across its rows)
                int cl = wn + j * 32 + 8 * q + 4 * hi;
                asm volatile("" : "+v"(cl));
                const float4_t mean = *(const float4_t *)(bnp + cl), sc = *(const float4_t *)(bnp + BN + cl),
                               sh = *(const float4_t *)(bnp + 2 * BN + cl);
#pragma unroll
                for(int e2 = 0; e2 < 2; e2++) {
                    const unsigned word = pk[i][j][2 * q + e2];
                    const h2 hv = __builtin_bit_cast(h2, word), xv = __builtin_bit_cast(h2, wx[side][2 * half + e2]);
                    unsigned keep = 0;
#pragma unroll
                    for(int h = 0; h < 2; h++) {
                        const int e = 2 * e2 + h;
                        const float xe = (float)xv[h];
                        const bool pos = !g.bq_relu || (float)(half_t)__builtin_fmaf(xe, sc[e], sh[e]) > 0.0f;
                        const bool on = ok && pos;
                        keep |= on ? (h ? 0xffff0000u : 0x0000ffffu) : 0u;
                        const float gv = on ? (float)hv[h] : 0.0f;
                        gf[side][e] = gv;
                        gq[side][e] = gv * (xe - mean[e]);
                    }
                    pk[i][j][2 * q + e2] = word & keep;
                }
            }
            // v_permlane16_swap exchanges the odd 16-lane rows of its first operand with the even rows of the
            // second: afterwards the two operands of a lane add up to what it keeps plus what its partner sent
#pragma unroll
            for(int e = 0; e < 4; e++) {
                const auto a = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, gf[0][e]),
                                                                __builtin_bit_cast(unsigned, gf[1][e]), false, false);
                const auto b = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, gq[0][e]),
                                                                __builtin_bit_cast(unsigned, gq[1][e]), false, false);
                // (the four results go through an opaque statement: hipcc 7.2 otherwise folds the sum of the
                // two results of one swap into twice the first)
                unsigned a0 = a[0], a1 = a[1], b0 = b[0], b1 = b[1];
                asm volatile("" : "+v"(a0), "+v"(a1), "+v"(b0), "+v"(b1));
                sv[4 * half + e] += __builtin_bit_cast(float, a0) + __builtin_bit_cast(float, a1);
                qv[4 * half + e] += __builtin_bit_cast(float, b0) + __builtin_bit_cast(float, b1);
            }
            // added here and now (left to itself the compiler postpones the additions to the end of the column
            // and keeps every exchanged value in a register until then)
#pragma unroll
            for(int e = 0; e < 4; e++)
                asm volatile("" : "+v"(sv[4 * half + e]), "+v"(qv[4 * half + e]));
            __builtin_amdgcn_sched_barrier(0);
        }
        // after the swaps: lower half-wave holds channels 0..7 (then 16..23) of the tile,
        // upper half-wave 8..15 (24..31): one store covers 32 contiguous bytes per pixel
        half_t *orow = g.out + pixr[i] * g.ldo;
#pragma unroll
        for(int q = 0; q < 2; q++) {
            const auto s0_ = __builtin_amdgcn_permlane32_swap(pk[i][j][4 * q + 0], pk[i][j][4 * q + 2], false, false);
            const auto s1_ = __builtin_amdgcn_permlane32_swap(pk[i][j][4 * q + 1], pk[i][j][4 * q + 3], false, false);
            const int n = nb + 16 * q + 8 * hi;
            if(ok && n < g.Ngemm) {
                const u4 o = {s0_[0], s1_[0], s0_[1], s1_[1]};
                *(u4 *)(orow + n) = o;
            }
        }
        if(i == TM - 1) {
            // lanes of a half-wave hold different pixels of the same 16 channels: after the remaining halving
            // exchanges each pair of lanes holds one channel's total over the wave tile's rows
            halve_exchange<8, 8>(sv, qv, lane);
            halve_exchange<4, 4>(sv, qv, lane);
            halve_exchange<2, 2>(sv, qv, lane);
            sres[j] = sv[0] + dpp_read<0xb1>(sv[0]);
            qres[j] = qv[0] + dpp_read<0xb1>(qv[0]);
        }
        __builtin_amdgcn_sched_barrier(0); // one sub-tile at a time: interleaving them costs registers
    }
    // pair p = (lane%32)/2 holds, per column j, channel 32*j + 8*(p/4) + 4*hi + p%4 of the wave tile;
    // the wavefronts stacked along M are added through LDS in a fixed order
    typedef float float2_t __attribute__((ext_vector_type(2)));
    float2_t *red = (float2_t *)smem;
    const int p = (lane & 31) >> 1;
    __syncthreads(); // every wavefront is done reading the last slice, which the sums below overwrite
    if((lane & 1) == 0) {
#pragma unroll
        for(int j = 0; j < TN; j++) {
            const float2_t v2 = {sres[j], qres[j]};
            red[(wave / WGN) * BN + wn + 32 * j + 8 * (p >> 2) + 4 * hi + (p & 3)] = v2;
        }
    }
    __syncthreads();
    if(tid < BN && n0 + tid < g.Ngemm) {
        float2_t t = red[tid];
#pragma unroll
        for(int wy = 1; wy < WGM; wy++)
            t += red[wy * BN + tid];
        *(float2_t *)(g.bq_partial + ((int64_t)stats_row * g.Ngemm + n0 + tid) * 2) = t;
    }
}

} // namespace
