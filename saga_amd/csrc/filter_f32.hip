// Backward filter of fp32 3x3, stride-1 convolutions on the bf16 matrix unit (split_f32.hpp), both operands split once per tile and
// not once per tap: dw[k][tap][c] = sum over pixels of dy[k][p] * x[c][p + tap].
//
// A persistent block owns 64 output x 64 input channels under all nine taps and walks tiles of 8x8 pixels of an image; a
// wavefront has 32 x 32 of them, the leading products and the small ones of every tap in registers (288 of the 512 that a lone
// wavefront of a SIMD may use).  Eight channels of a position are loaded (one lane each), split and left in LDS as 16 bytes
// per part: x with a border of one, and dy.  The reduction index of a matrix instruction is the pixel, eight columns of two rows,
// one row per half of the wavefront, from the transposing LDS read; a tile is walked downwards, so that rows (2j, 2j+1) of
// x are the operand of the top taps in one step and were that of the bottom taps in the one before: 7 operands of three parts
// for 54 instructions, 0.39 KB of LDS per instruction.
// Loads, splitting and LDS writes of the next tiles go out between the instructions; three pieces of eight loads per lane are on
// their way at any time.
// Slots are 128 bytes; their 16-byte chunks are swizzled by the column, bit 2 by pairs of columns, which spreads a read (four
// columns, 32 channels) over all banks, the lower bits by fours, which do the same for a write (sixteen columns, one chunk).
//
// Where 32 channels of a kind are all there are, a block has 32 of them, and its wavefronts share the steps of a tile (of 16 rows, if
// both are few) and add up their sums in LDS in the end; with 64 three of four wavefronts multiplied zeros.  us, both launches, before
// -> now: 16->16 at 512x32x32 162 -> 63, at 128x32x32 50 -> 27, 24->24 at 16x112x112 69 -> 36, 32->32 at 512x16x16 51 -> 30, 32->64 at 32x56x56 51 ->
// 41, 128->16 at 70x24x24 39 -> 32.  A tile takes 2.9 us of which the matrix instructions are 1.5: what bounds them is loading, four
// bytes at a time, and splitting.
//
// Tiles overlap where they do not divide an image, with zeros for the gradients of pixels seen before.  A sum that is not
// finite had an operand without three parts: its block takes its share again in fp32 products.
#include "split_f32.hpp"
#include "filter_f32.hpp"

#include <algorithm>
#include <type_traits>

namespace {

typedef short short4_t __attribute__((ext_vector_type(4)));
typedef short short8_t __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) void *lds_ptr_t;

struct WindowFilterArgs {
    const float *x, *dy;
    float *partial;
    long long x_sn, x_sc, x_sh, x_sw, y_sn, y_sc, y_sh, y_sw;
    unsigned x_bytes, y_bytes; // of one image
    int H, W, C, K;
    int nx, tpi, ntiles;
    int pairs, pairs_c, splits;
};

constexpr unsigned OOB = 0x7fffff00u;
constexpr int TILE = 8, SR = TILE + 2, TAPS = 9;

// A block: 32 * WK output and 32 * WC input channels, of which FILLED (of 32) are loaded, tiles of 8 columns and ROWS rows; the
// wavefronts that do not have channels of their own share a tile's steps of two rows.
template <int WK, int WC, int ROWS, int FILLED> struct Block {
    static constexpr int KB = 32 * WK, CB = 32 * WC, ROWS_X = ROWS + 2, SHARE = 4 / (WK * WC), STEPS = ROWS / 2 / SHARE, GROUPS = 3 * STEPS;
    static constexpr int XSLOT = 2 * CB, YSLOT = 2 * KB; // bytes of a position's channels, of one part
    static constexpr int NOWHERE = ROWS_X * SR * XSLOT, XPART = NOWHERE + (SHARE > 1 ? 128 : 0), YPART = ROWS * TILE * YSLOT, BUFFER = 3 * (XPART + YPART);
    static constexpr int SUMS = SHARE > 1 ? 4 * TAPS * 16 * 64 * 4 : 0; // what the wavefronts add up in the end
    static constexpr int LDS = std::max(2 * BUFFER, SUMS);
    static constexpr int XCHUNKS = FILLED * WC / 8, YCHUNKS = FILLED * WK / 8;
    // pieces of a tile, and those on their way: one divides the other, that a piece's registers are always the same ones
    static constexpr int XITEMS = (ROWS_X * SR * XCHUNKS + 255) / 256, ITEMS = XITEMS + ROWS * TILE * YCHUNKS / 256, RING = SHARE > 1 ? ITEMS : 3;
    static_assert(STEPS * 2 * SHARE == ROWS && ROWS * TILE * YCHUNKS % 256 == 0 && ITEMS <= GROUPS && ITEMS % RING == 0 && LDS <= 160 * 1024, "");
};

// (of 64 channels' eight chunks; 32 channels' four take up all banks with the columns that are read together, and are only spread for
// the writes)
template <int SLOT> __device__ __forceinline__ int chunk_swizzle(int col)
{
    return SLOT == 128 ? ((col >> 1) & 1) << 2 | ((col >> 2) & 1) << 1 | ((col >> 3) & 1) : (col >> 2) & 3;
}

// 8 pixels of one channel from the two addresses' fours; the caller waits (the compiler does not know that these read LDS)
template <int OFF> __device__ __forceinline__ bf16x8_t read_pixels(unsigned lo, unsigned hi)
{
    short4_t a, b;
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(a) : "v"(lo), "n"(OFF) : "memory");
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(b) : "v"(hi), "n"(OFF) : "memory");
    return __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

// some taps' sums, from `tap` on
template <int N> __device__ __forceinline__ void store_sums(const WindowFilterArgs &t, int split, int k, int c, int tap, const float16_t (&acc)[N])
{
    // (a share's partial result is one buffer: rows and columns beyond the filter are outside)
    const unsigned bytes = (unsigned)t.K * (TAPS * 4u) * (unsigned)t.C, krow = TAPS * 4u * (unsigned)t.C;
    const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc((void *)((char *)t.partial + (int64_t)split * bytes), 0, bytes, 0x00020000);
    const unsigned first = c < t.C ? (unsigned)k * krow + (unsigned)c * 4u : OOB;
#pragma unroll
    for(int i = 0; i < N; i++)
#pragma unroll
        for(int v = 0; v < 16; v++) {
            const float sum = acc[i][v]; // (the cast takes a vector's element for its first)
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, sum), ro, first + (8 * (v / 4) + v % 4) * krow,
                                                  (tap + i) * t.C * 4, 0);
        }
}

// A block's share in fp32 products: a tile's pixels of x, with a border of one, and of dy go to LDS as they are, a matrix
// instruction takes two neighbouring pixels, the next tile's loads are on their way meanwhile.  us, second pass included, finite / one
// NaN (a wavefront's share pixel by pixel, as it was): 64->64 at 256x56x56 311 / 1110 (3320), 512->512 at 9x8x8 50 / 102 (222); the
// kernel for fp32 matrix instructions 580 and 68.
template <int WK, int WC, int ROWS, int FILLED>
__device__ __forceinline__ void windows_again(const WindowFilterArgs &t, int split, int k0, int c0, int mt, int nt, int part, float16_t (&acc)[TAPS],
                                              char *smem)
{
    typedef Block<WK, WC, ROWS, FILLED> B;
    constexpr int XPOS = B::ROWS_X * SR, YPOS = ROWS * TILE, XPITCH = XPOS + 1, YPITCH = YPOS + 1; // of a channel; odd, for the banks
    static_assert((B::CB * XPITCH + B::KB * YPITCH) * 4 <= B::LDS, "");
    float *const xs = (float *)smem, *const ys = xs + B::CB * XPITCH;
    const int tid = threadIdx.x, lane = tid & 63, hi = lane >> 5;
#pragma unroll
    for(int tp = 0; tp < TAPS; tp++)
#pragma unroll
        for(int v = 0; v < 16; v++)
            acc[tp][v] = 0.0f;
    constexpr int XN = (B::CB * XPOS + 255) / 256, YN = B::KB * YPOS / 256;
    static_assert(YN * 256 == B::KB * YPOS, "whole rounds");
    const unsigned xrange = t.x_bytes - (unsigned)(c0 * t.x_sc * 4), yrange = t.y_bytes - (unsigned)(k0 * t.y_sc * 4);
    struct Tile {
        int n, ox, oy, dup_cols, dup_rows;
    };
    auto place = [&](int tile) {
        const int n = tile / t.tpi, in = tile - n * t.tpi, ty = in / t.nx, tx = in - ty * t.nx;
        const int ox = std::min(tx * TILE, t.W - TILE), oy = std::min(ty * ROWS, t.H - ROWS);
        return Tile{n, ox, oy, tx * TILE - ox, ty * ROWS - oy};
    };
    float xr[XN], yr[YN]; // the next tile's
    auto load = [&](const Tile &p) {
        const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void *)(t.x + p.n * t.x_sn + c0 * t.x_sc), 0, xrange, 0x00020000);
        const __amdgpu_buffer_rsrc_t ry = __builtin_amdgcn_make_buffer_rsrc((void *)(t.dy + p.n * t.y_sn + k0 * t.y_sc), 0, yrange, 0x00020000);
#pragma unroll
        for(int u = 0; u < XN; u++) {
            const int i = u * 256 + tid, ch = i / XPOS, pos = i - ch * XPOS, iy = p.oy + pos / SR - 1, ix = p.ox + pos % SR - 1;
            const bool there = ch < B::CB && c0 + ch < t.C && (unsigned)iy < (unsigned)t.H && (unsigned)ix < (unsigned)t.W;
            xr[u] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                  rx, there ? (unsigned)((ch * t.x_sc + iy * t.x_sh + ix * t.x_sw) * 4) : OOB, 0, 0));
        }
#pragma unroll
        for(int u = 0; u < YN; u++) {
            const int i = u * 256 + tid, ch = i / YPOS, pos = i % YPOS, iy = p.oy + pos / TILE, ix = p.ox + pos % TILE;
            yr[u] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                  ry, k0 + ch < t.K ? (unsigned)((ch * t.y_sc + iy * t.y_sh + ix * t.y_sw) * 4) : OOB, 0, 0));
        }
    };
    Tile p = place(split);
    load(p);
#pragma unroll 1
    for(int tile = split; tile < t.ntiles; tile += t.splits) {
        __syncthreads();
#pragma unroll
        for(int u = 0; u < XN; u++)
            if(u * 256 + tid < B::CB * XPOS)
                xs[(u * 256 + tid) / XPOS * XPITCH + (u * 256 + tid) % XPOS] = xr[u];
#pragma unroll
        for(int u = 0; u < YN; u++)
            ys[(u * 256 + tid) / YPOS * YPITCH + (u * 256 + tid) % YPOS] = yr[u];
        __syncthreads();
        const int dup_cols = p.dup_cols, dup_rows = p.dup_rows; // that a tile before had: both operands zero
        p = place(tile + t.splits < t.ntiles ? tile + t.splits : tile);
        load(p);
        const float *const xc = xs + (nt * 32 + (lane & 31)) * XPITCH, *const yc = ys + (mt * 32 + (lane & 31)) * YPITCH;
#pragma unroll 1
        for(int row = std::max(dup_rows, 2 * B::STEPS * part); row < 2 * B::STEPS * (part + 1); row++)
#pragma unroll
            for(int two = 0; two < TILE; two += 2) {
                const int col = two + hi;
                const bool own = col >= dup_cols;
                const float g = own ? yc[row * TILE + col] : 0.0f;
#pragma unroll
                for(int tp = 0; tp < TAPS; tp++)
                    acc[tp] = __builtin_amdgcn_mfma_f32_32x32x2f32(g, own ? xc[(row + tp / 3) * SR + col + tp % 3] : 0.0f, acc[tp], 0, 0, 0);
            }
    }
}

template <int WK, int WC, int ROWS, int FILLED>
__global__ void __launch_bounds__(256, 1) conv_f32_bwd_filter_windows(WindowFilterArgs t)
{
    typedef Block<WK, WC, ROWS, FILLED> B;
    constexpr int ITEMS = B::ITEMS, XITEMS = B::XITEMS, XPART = B::XPART, YPART = B::YPART;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63, hi = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int mt = wave / WC % WK, nt = wave % WC, part = wave / (WK * WC);
    const int b0 = xcd_remap(blockIdx.x, gridDim.x);
    const int split = __builtin_amdgcn_readfirstlane(b0 / t.pairs), pair = b0 - split * t.pairs;
    const int kb = __builtin_amdgcn_readfirstlane(pair / t.pairs_c), k0 = kb * B::KB, c0 = (pair - kb * t.pairs_c) * B::CB;

    // This lane's pieces: offset of the position's first channel from the tile's first pixel (x: from the one left of and above it),
    // where it goes in LDS, and one bit per piece that reads zeros: always, at an image's left, right, upper, lower
    // border, in tiles that overlap.
    unsigned roff[ITEMS], slot[ITEMS];
    unsigned dead = 0, left = 0, right = 0, top = 0, bottom = 0, cols = 0, rows = 0;
    const int dup_cols = t.nx * TILE - t.W, dup_rows = t.tpi / t.nx * ROWS - t.H;
#pragma unroll
    for(int u = 0; u < ITEMS; u++) {
        const bool is_x = u < XITEMS;
        const int wide = is_x ? SR : TILE, all = is_x ? B::ROWS_X * SR : ROWS * TILE, L = (is_x ? u : u - XITEMS) * 256 + tid, g = L / all, pos = L - g * all;
        const int r = pos / wide, col = pos - r * wide;
        if(is_x) {
            roff[u] = (unsigned)((r * t.x_sh + col * t.x_sw + g * 8 * t.x_sc) * 4);
            dead |= g >= B::XCHUNKS || c0 + 8 * g >= t.C ? 1u << u : 0u;
            left |= col == 0 ? 1u << u : 0u;
            right |= col == SR - 1 ? 1u << u : 0u;
            top |= r == 0 ? 1u << u : 0u;
            bottom |= r == B::ROWS_X - 1 ? 1u << u : 0u;
        } else {
            roff[u] = (unsigned)((r * t.y_sh + col * t.y_sw + g * 8 * t.y_sc) * 4);
            dead |= k0 + 8 * g >= t.K ? 1u << u : 0u;
            cols |= col < dup_cols ? 1u << u : 0u;
            rows |= r < dup_rows ? 1u << u : 0u;
        }
        // (lanes of x without a position write nothing, or behind the part)
        const int chunk = is_x ? g ^ chunk_swizzle<B::XSLOT>(col) : g ^ chunk_swizzle<B::YSLOT>(col);
        slot[u] = g < (is_x ? B::XCHUNKS : B::YCHUNKS) ? (unsigned)((is_x ? 0 : 3 * XPART) + pos * (is_x ? B::XSLOT : B::YSLOT) + (chunk << 4)) : B::SHARE > 1 ? B::NOWHERE : 0xffffffffu;
    }
    struct Tile {
        const float *x, *y;
        unsigned xbase, ybase, kill;
    };
    auto place = [&](int tile) { // (behind the last tile: zeros, that the number of loads does not depend on it)
        Tile r;
        const bool real = tile < t.ntiles;
        const int tl = real ? tile : 0, n = __builtin_amdgcn_readfirstlane(tl / t.tpi), in = tl - n * t.tpi;
        const int ty = __builtin_amdgcn_readfirstlane(in / t.nx), tx = in - ty * t.nx;
        const int ox = std::min(tx * TILE, t.W - TILE), oy = std::min(ty * ROWS, t.H - ROWS);
        r.x = t.x + n * t.x_sn + c0 * t.x_sc;
        r.y = t.dy + n * t.y_sn + k0 * t.y_sc;
        r.xbase = (unsigned)(((oy - 1) * t.x_sh + (ox - 1) * t.x_sw) * 4);
        r.ybase = (unsigned)((oy * t.y_sh + ox * t.y_sw) * 4);
        r.kill = dead | (ox == 0 ? left : 0u) | (ox + TILE == t.W ? right : 0u) | (oy == 0 ? top : 0u) | (oy + ROWS == t.H ? bottom : 0u) |
                 (ox < tx * TILE ? cols : 0u) | (oy < ty * ROWS ? rows : 0u);
        if(!real)
            r.kill = 0xffffffffu;
        return r;
    };
    const unsigned xrange = t.x_bytes - (unsigned)(c0 * t.x_sc * 4), yrange = t.y_bytes - (unsigned)(k0 * t.y_sc * 4);
    float ring[B::RING][8];
    auto load_piece = [&](const Tile &r, auto U) {
        constexpr int u = U.value;
        constexpr bool is_x = u < XITEMS;
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)(is_x ? r.x : r.y), 0, is_x ? xrange : yrange, 0x00020000);
        const unsigned off = (roff[u] + (is_x ? r.xbase : r.ybase)) | ((r.kill << (31 - u)) & 0x80000000u);
        const unsigned step = (unsigned)((is_x ? t.x_sc : t.y_sc) * 4);
#pragma unroll
        for(int j = 0; j < 8; j++)
            ring[u % B::RING][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, off, j * step, 0));
    };
    auto write_piece = [&](char *to, auto U) {
        constexpr int u = U.value, part_bytes = u < XITEMS ? XPART : YPART;
        Parts p;
        split3(ring[u % B::RING], p);
        // (a branch where a tile has few steps costs 400 spilled registers, none where it has four 5 % of the time)
        if(B::SHARE > 1 || u != XITEMS - 1 || slot[u] != 0xffffffffu) {
#pragma unroll
            for(int h = 0; h < 3; h++)
                *(uint4_t *)(to + slot[u] + h * part_bytes) = p.v[h];
        }
    };

    // Operand addresses: a lane of a transposing read points at column fp (second half: fp + 4) of its row and four channels.
    const int fp = (lane & 15) >> 2, fc = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
    const unsigned lds0 = (unsigned)(uintptr_t)(lds_ptr_t)smem;
    unsigned xa[3][2], ya[2];
    auto at = [&](auto SLOT, int wide, int col, int ch) {
        constexpr int slot_bytes = SLOT.value;
        return (unsigned)((2 * B::STEPS * part + hi) * wide * slot_bytes + col * slot_bytes + (((ch >> 3) ^ chunk_swizzle<slot_bytes>(col)) << 4) + (ch & 7) * 2);
    };
#pragma unroll
    for(int e = 0; e < 2; e++) {
#pragma unroll
        for(int s = 0; s < 3; s++)
            xa[s][e] = lds0 + at(std::integral_constant<int, B::XSLOT>(), SR, fp + s + 4 * e, nt * 32 + fc);
        ya[e] = lds0 + 3 * XPART + at(std::integral_constant<int, B::YSLOT>(), TILE, fp + 4 * e, mt * 32 + fc);
    }

    float16_t acc[TAPS], low[TAPS];
#pragma unroll
    for(int tp = 0; tp < TAPS; tp++)
#pragma unroll
        for(int v = 0; v < 16; v++)
            acc[tp][v] = low[tp][v] = 0.0f;

    if constexpr(FILLED < 32) { // channels that nobody loads: zeros, once
        for(int i = tid; i < 2 * B::BUFFER / 16; i += 256)
            ((uint4_t *)smem)[i] = uint4_t{0, 0, 0, 0};
        __syncthreads();
    }
    int tile = split, b = 0;
    Tile next = place(tile + t.splits);
    {
        const Tile first = place(tile);
        each<0, B::RING>([&](auto U) { load_piece(first, U); });
        each<0, ITEMS>([&](auto U) {
            write_piece(smem, U);
            if constexpr(U.value + B::RING < ITEMS)
                load_piece(first, std::integral_constant<int, U.value + B::RING>());
            else
                load_piece(next, std::integral_constant<int, U.value + B::RING - ITEMS>());
        });
    }
#pragma unroll 1
    for(; tile < t.ntiles; tile += t.splits) {
        // everybody's share of this tile is there, and everybody is done with the other buffer
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        const Tile after = place(tile + 2 * t.splits);
        char *const to = smem + (b ^ 1) * B::BUFFER;
        unsigned xs[3][2], ys[2];
#pragma unroll
        for(int e = 0; e < 2; e++) {
#pragma unroll
            for(int s = 0; s < 3; s++)
                xs[s][e] = xa[s][e] + b * B::BUFFER;
            ys[e] = ya[e] + b * B::BUFFER;
        }
        bf16x8_t even[3][3], odd[3][3], grad[2][3]; // [column of the tap][part]
        auto read_x = [&](bf16x8_t(&to)[3][3], auto ROW) {
            each<0, 9>([&](auto I) {
                constexpr int s = I.value / 3, h = I.value % 3;
                to[s][h] = read_pixels<ROW.value * SR * B::XSLOT + h * XPART>(xs[s][0], xs[s][1]);
            });
        };
        auto read_grad = [&](auto J) {
            each<0, 3>([&](auto H) { grad[J.value & 1][H.value] = read_pixels<J.value * 2 * TILE * B::YSLOT + H.value * YPART>(ys[0], ys[1]); });
        };
        auto there = [&](bf16x8_t(&x)[3][3], bf16x8_t(&g)[3]) { // (the multiplications stay behind the wait: their operands pass through it)
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
            for(int s = 0; s < 3; s++) {
                asm volatile("" : "+v"(x[s][0]), "+v"(x[s][1]), "+v"(x[s][2]));
                asm volatile("" : "+v"(g[s]));
            }
        };
        read_grad(std::integral_constant<int, 0>());
        read_x(even, std::integral_constant<int, 0>());
        // group G: the three taps of filter row G % 3 in step G / 3
        each<0, B::GROUPS>([&](auto G) {
            constexpr int j = G.value / 3, row = G.value % 3;
            constexpr int u = std::min((G.value * ITEMS + B::GROUPS - 1) / B::GROUPS, ITEMS - 1); // the piece of this group, if it has one
            bf16x8_t(&x)[3][3] = row == 1 ? odd : even;
            bf16x8_t(&g)[3] = grad[j & 1];
            there(x, g);
            // what the next group needs
            if constexpr(row == 0)
                read_x(odd, std::integral_constant<int, 2 * j + 1>());
            if constexpr(row == 1)
                read_x(even, std::integral_constant<int, 2 * j + 2>());
            if constexpr(row == 2 && j + 1 < B::STEPS)
                read_grad(std::integral_constant<int, j + 1>());
            __builtin_amdgcn_sched_barrier(0);
            each<0, SPLIT_PRODUCTS>([&](auto P) {
                constexpr int qi[] = {0, 1, 0, 1, 2, 0}, pi[] = {0, 0, 1, 1, 0, 2};
                each<0, 3>([&](auto S) {
                    constexpr int tp = row * 3 + S.value;
                    bf16x8_t &q = g[qi[P.value]], &p = x[S.value][pi[P.value]];
                    float16_t &sum = P.value ? low[tp] : acc[tp];
                    // (of its own accord the compiler gives sums only the 256 accumulation registers, sixteen of these eighteen)
                    if constexpr(tp == 8)
                        asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(sum) : "v"(q), "v"(p));
                    else if constexpr(B::SHARE > 1) // (here a dozen of them would be spilled)
                        asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(sum) : "v"(q), "v"(p));
                    else
                        sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(q, p, sum, 0, 0, 0);
                });
                if constexpr(u * B::GROUPS / ITEMS == G.value && P.value == 2) {
                    write_piece(to, std::integral_constant<int, u>());
                    load_piece(u + B::RING < ITEMS ? next : after, std::integral_constant<int, (u + B::RING) % ITEMS>());
                }
            });
            __builtin_amdgcn_sched_barrier(0);
        });
        next = after;
        b ^= 1;
    }
    // (the products of the last instructions are on their way, and the compiler knows only of its own)
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
    for(int tp = 0; tp < TAPS; tp++)
        if(tp == 8)
            asm volatile("" : "+v"(acc[tp]), "+v"(low[tp]));
        else if(B::SHARE > 1)
            asm volatile("" : "+a"(acc[tp]), "+a"(low[tp]));

    float bad = 0.0f;
#pragma unroll
    for(int tp = 0; tp < TAPS; tp++)
#pragma unroll
        for(int v = 0; v < 16; v++) {
            acc[tp][v] = (acc[tp][v] + low[tp][v]) * SPLIT_SUM;
            bad = __builtin_fmaf(acc[tp][v], 0.0f, bad);
        }
    // (everybody's writes of a tile behind the last are done)
    volatile int *const found = (volatile int *)smem;
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    found[wave] = __builtin_amdgcn_ballot_w64(bad != bad) != 0;
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    // acc[tap][v]: output channel 8 * (v / 4) + v % 4 of a half's
    const int k = k0 + mt * 32 + 4 * hi, c = c0 + nt * 32 + (lane & 31);
    if(found[0] | found[1] | found[2] | found[3]) {
#pragma unroll
        for(int tp = 0; tp < TAPS; tp++)
#pragma unroll
            for(int v = 0; v < 16; v++)
                acc[tp][v] = 0.0f;
        windows_again<WK, WC, ROWS, FILLED>(t, split, k0, c0, mt, nt, part, acc, smem);
        if constexpr(B::SHARE == 1)
            store_sums(t, split, k, c, 0, acc);
    } else if constexpr(B::SHARE == 1) {
        store_sums(t, split, k, c, 0, acc);
    }
    if constexpr(B::SHARE > 1) {
        // the sums of the wavefronts that shared the pixels meet in LDS, in a fixed order; each stores some of the taps
        float4_t *const sums = (float4_t *)smem; // [tap][four][wavefront][lane]
        __syncthreads();
#pragma unroll
        for(int tp = 0; tp < TAPS; tp++)
#pragma unroll
            for(int q = 0; q < 4; q++)
                sums[((tp * 4 + q) * 4 + wave) * 64 + lane] = float4_t{acc[tp][4 * q], acc[tp][4 * q + 1], acc[tp][4 * q + 2], acc[tp][4 * q + 3]};
        __syncthreads();
        for(int tp = part; tp < TAPS; tp += B::SHARE) {
            float16_t sum[1];
#pragma unroll
            for(int q = 0; q < 4; q++) {
                float4_t f = {0, 0, 0, 0};
#pragma unroll
                for(int h = 0; h < B::SHARE; h++)
                    f += sums[((tp * 4 + q) * 4 + h * (4 / B::SHARE) + wave % (4 / B::SHARE)) * 64 + lane];
#pragma unroll
                for(int e = 0; e < 4; e++)
                    sum[0][4 * q + e] = f[e];
            }
            store_sums(t, split, k, c, tp, sum);
        }
    }
}

// bytes of one image, or 0
unsigned image_bytes(const SagaTensorView *v)
{
    long long last = 0;
    for(int i = 1; i < 4; i++) {
        if(v->strides[i] < 0)
            return 0;
        last += (v->dims[i] - 1ll) * v->strides[i];
    }
    return last * 4 + 4 < 0x7fff0000ll ? (unsigned)(last * 4 + 4) : 0;
}

} // namespace

// Where a block walks three tiles or more, and where that takes less time than the kernels for fp32 matrix instructions, which have
// fewer pixels outside small images and fewer channels that are not there.  us, the kernel for fp32 matrix instructions (conv_f32_bwd_filter_uniform, where channels come
// in 32s) / this one, both with the second pass:
//   64->64   256x56x56  581 / 312   128->128 64x28x28  169 / 114   512->512  8x28x28  355 / 207   96->160 32x40x40    189 / 124
//   64->64    64x56x56  178 /  95   256->256 128x14x14 311 / 192   32->32  128x16x16   46 /  37   16->16  128x32x32    67 /  51
//   64->64    16x56x56   59 /  45   256->256  32x14x14  96 /  64   72->136   9x29x17   41 /  35   8->24    64x32x32    31 /  31
// and left to them: 16->128 225x9x9 31 / 48, 32->104 130x11x11 27 / 39, 8->416 78x12x12 38 / 53, 64->120 76x11x11 32 / 41.  Of the 221
// layers the slower kernel is taken in two, by 5 and 8 %.
// 312 us are 190 TFLOP/s of fp32 work, 1140 of bf16: what bounds it is the matrix unit, and the reading of operands for the first step of
// a tile, which nothing hides.  Relative error against 64 bits, the same shapes: 4.3e-7 to 9.8e-7 before, 1.2e-7 to 2.5e-7.
FilterWindows plan_filter_windows(const ConvGeom &g)
{
    if(g.R != 3 || g.S != 3 || g.stride != 1 || g.pad != 1 || g.dil != 1 || g.group != 1 || g.P != g.H || g.Q != g.W || g.W < TILE ||
       g.H < TILE || g.K % 8 || g.C % 8 || (long long)g.K * g.C * TAPS * 4 >= 0x7fff0000ll)
        return {};
    FilterWindows p;
    const bool few_k = g.K <= 32, few_c = g.C <= 32 && !(few_k && g.H < 16);
    p.kb = few_k ? 32 : 64;
    p.cb = few_c ? 32 : 64;
    p.rows = few_k && few_c ? 16 : TILE;
    const int64_t pairs = (int64_t)((g.K + p.kb - 1) / p.kb) * ((g.C + p.cb - 1) / p.cb);
    const int64_t tiles = (int64_t)((g.W + TILE - 1) / TILE) * ((g.H + p.rows - 1) / p.rows) * g.N;
    int64_t share = std::max<int64_t>(1, 256 / pairs);
    if(few_k || few_c)
        share = std::max<int64_t>(1, std::min(share, tiles / 3));
    if(pairs > 1024 || tiles >= 0x7fffffff || tiles < 2 * share + 1)
        return {};
    p.pairs = (int)pairs;
    p.splits = (int)share;
    p.tiles = (int)tiles;
    return p;
}

// Both launches and the first tile, tiles of a block one after the other, and partial results to write and add up (fitted to 221 layers of 8
// to 512 channels, 16 % off at most; with 32 channels of a kind in a block to 11 layers, 10 %).
double filter_windows_ns(const FilterWindows &p, const ConvGeom &g)
{
    const bool whole = p.kb == 64 && p.cb == 64;
    return (whole ? 9500 : 13400) + (whole ? 4430.0 : p.rows == TILE ? 2450.0 : 2850.0) * ((p.tiles + p.splits - 1) / p.splits) +
           2.24e-3 * p.splits * g.K * g.C * TAPS;
}

template <int WK, int WC, int ROWS, int FILLED = 32> static int launch(const WindowFilterArgs &t, hipStream_t st)
{
    constexpr int room = Block<WK, WC, ROWS, FILLED>::LDS;
    static const hipError_t allowed =
        hipFuncSetAttribute((const void *)conv_f32_bwd_filter_windows<WK, WC, ROWS, FILLED>, hipFuncAttributeMaxDynamicSharedMemorySize, room);
    if(allowed != hipSuccess)
        return (int)allowed;
    conv_f32_bwd_filter_windows<WK, WC, ROWS, FILLED><<<t.pairs * t.splits, 256, room, st>>>(t);
    SAGA_CHECK_LAUNCH();
    return 0;
}

int launch_filter_windows(const FilterWindows &p, const SagaTensorView *x, const SagaTensorView *dy, float *partial, const ConvGeom &g,
                          hipStream_t st)
{
    WindowFilterArgs t;
    t.x_bytes = image_bytes(x);
    t.y_bytes = image_bytes(dy);
    if(!t.x_bytes || !t.y_bytes)
        return SAGA_HIP_EUNSUPPORTED;
    t.x = (const float *)x->ptr;
    t.dy = (const float *)dy->ptr;
    t.partial = partial;
    t.x_sn = x->strides[0]; t.x_sc = x->strides[1]; t.x_sh = x->strides[2]; t.x_sw = x->strides[3];
    t.y_sn = dy->strides[0]; t.y_sc = dy->strides[1]; t.y_sh = dy->strides[2]; t.y_sw = dy->strides[3];
    t.H = g.H;
    t.W = g.W;
    t.C = g.C;
    t.K = g.K;
    t.nx = (g.W + TILE - 1) / TILE;
    t.tpi = t.nx * ((g.H + p.rows - 1) / p.rows);
    t.ntiles = p.tiles;
    t.pairs = p.pairs;
    t.pairs_c = (g.C + p.cb - 1) / p.cb;
    t.splits = p.splits;
    if(p.kb == 64)
        return p.cb == 64 ? launch<2, 2, 8>(t, st) : launch<2, 1, 8>(t, st);
    return p.cb == 64 ? launch<1, 2, 8>(t, st) : t.K <= 16 && t.C <= 16 ? launch<1, 1, 16, 16>(t, st) : launch<1, 1, 16>(t, st);
}
