// Backward filter of 3x3, stride-1 convolutions over images: dw[k][tap][c] = sum over pixels of dy[p][k] * x[p + tap][c].
//
// A persistent block owns 64 output x 64 input channels under all nine taps and walks tiles of an image: the tile's pixels of
// dy and, with a border of one, of x are copied once to LDS, the next tile's while this one is multiplied.  Two groups of two
// wavefronts share a tile's pixels: a wavefront has 32 of the input channels, all 64 output channels, and the whole of
// their nine taps in registers (288 of the 512 that a lone wavefront of a SIMD may use); the groups' sums meet in LDS
// at the end.  One partial result per block goes to the second pass.
//
// The reduction index of a matrix instruction is the pixel, sixteen of them: eight columns (a group's strip) of two rows, one row
// per half of the wavefront, from the transposing LDS read.  A strip is walked downwards: of x, rows (2j, 2j+1) are the
// operand of the top taps in step j and of the bottom taps in the step before, rows (2j+1, 2j+2) that of the middle taps.  So
// a step of 18 instructions reads 6 operands of x and 2 of dy: with an operand of its own for every tap, and half as many output
// channels per wavefront, it were 20, and the LDS, not the matrix unit, the bound.
// Pixel slots are 128 bytes, their 16-byte chunks swizzled by the column: 32 lanes of a read (four columns, 32 channels) then
// hit 64 banks, and as the width of a tile is known here, every read is an immediate offset from five addresses.
//
// Tiles overlap at the right and the lower border of an image that they do not divide; pixels seen before have zeros
// for dy.  An infinity of x there makes a NaN of a sum that should be infinite: a block that ends with a NaN looks for
// one, and if there is one takes its share again, with zeros for x as well.
#include "filter_strips.hpp"

#include <algorithm>
#include <type_traits>

namespace {

typedef short short4_t __attribute__((ext_vector_type(4)));
typedef unsigned uint4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void *lds_ptr_t;

struct StripArgs {
    const half_t *x, *dy;
    float *partial; // [split][K][9][C]
    int ldx, ldy, H, W, C, K;
    int nx, tpi, ntiles; // tiles of a row of them, of an image, of all
    int pairs, pairs_c, splits;
};

// 8 pixels of one channel: instructions that the compiler does not know to read LDS (it would wait for every load into LDS that is
// on its way, the next tile's too).  The caller waits.
template <int LO> __device__ __forceinline__ half8_t read_pixels(unsigned addr)
{
    short4_t a, b;
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(a) : "v"(addr), "n"(LO) : "memory");
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(b) : "v"(addr), "n"(LO + 512) : "memory");
    return __builtin_bit_cast(half8_t, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

// The order of a tile's work: instruction 18 * j + m multiplies, in step j, x operand m % 6 / 2 (the tap's column) of the top (m < 6),
// middle and bottom taps with half m % 2 of dy.  Operands are read in the order of their first use, AHEAD instructions early.
constexpr int AHEAD = 8;
constexpr unsigned OOB = 0x7fffff00u; // behind every buffer: loads return zero, stores do nothing
constexpr int first_uses(int t, int nst)
{
    const int j = t / 18, m = t % 18;
    if(j >= nst)
        return 0;
    return (m < 2 ? 1 : 0) + (j == 0 && m < 6 && m % 2 == 0 ? 1 : 0) + (m >= 6 && m % 2 == 0 ? 1 : 0);
}
constexpr int reads_behind(int t, int nst) // those on their way behind the operands of instruction t
{
    int n = 0;
    for(int u = t + 1; u <= t + AHEAD; u++)
        n += first_uses(u, nst);
    return n;
}

template <int TW, int NST> struct StripTile {
    static constexpr int GROUP_ROWS = TW == 16 ? 0 : 2 * NST, TR = 2 * NST + GROUP_ROWS, SR = TW + 2;
    static constexpr int NLX = ((TR + 2) * SR * 8 + 255) / 256, NLY = TR * TW * 8 / 256;
    static constexpr int XB = NLX * 4096, YB = NLY * 4096;
    static constexpr int LDS = std::max(2 * (XB + YB), 4 * 36 * 1024); // (the groups' sums: half of a wavefront's accumulators)
    static_assert(TR * TW * 8 % 256 == 0 && LDS <= 160 * 1024 && NLX + NLY < 32, "tile");
};

// whether an infinity of x, in the block's channels from c0 on, is seen by pixels of its tiles that another tile has too (or by those next to them)
template <int TW, int TR> __device__ __forceinline__ bool infinity_under_overlap(const StripArgs &t, int split, int c0)
{
    bool found = false;
#pragma unroll 1
    for(int tile = split; tile < t.ntiles; tile += t.splits) {
        const int n = tile / t.tpi, in = tile - n * t.tpi, ty = in / t.nx, tx = in - ty * t.nx;
        const int ox = std::min(tx * TW, t.W - TW), oy = std::min(ty * TR, t.H - TR);
        if(ox == tx * TW && oy == ty * TR)
            continue;
        const half_t *const img = t.x + (int64_t)n * t.H * t.W * t.ldx + c0;
#pragma unroll 4
        for(int i = threadIdx.x; i < (TR + 2) * (TW + 2) * 8; i += 256) {
            const int pos = i >> 3, ch = (i & 7) * 8, y = oy + pos / (TW + 2) - 1, x = ox + pos % (TW + 2) - 1;
            if(ch < t.C - c0 && (unsigned)y < (unsigned)t.H && (unsigned)x < (unsigned)t.W) {
                const uint4_t v = *(const uint4_t *)(img + ((int64_t)y * t.W + x) * t.ldx + ch);
#pragma unroll
                for(int j = 0; j < 4; j++)
                    found |= (v[j] & 0x7fffu) == 0x7c00u || (v[j] & 0x7fff0000u) == 0x7c000000u;
            }
        }
    }
    return found;
}

// A block's share once more, straight from memory: a wavefront's 32 output channels from k0 on, this lane's input channel c.
// (us, second pass included, 192->192 at 15x23x19 / 512->512 at 9x17x33: finite 31 / 67, one NaN 41 / 99, one infinity
// under an overlap 83 / 262.)
template <int TW, int TR> __device__ __forceinline__ void strips_again(const StripArgs &t, int split, int k0, int c, __amdgpu_buffer_rsrc_t ro)
{
    const int lane = threadIdx.x & 63, hi = lane >> 5, k = k0 + (lane & 31);
    const int64_t ximg = (int64_t)t.H * t.W * t.ldx, yimg = (int64_t)t.H * t.W * t.ldy;
    float16_t acc[9];
#pragma unroll
    for(int tp = 0; tp < 9; tp++)
#pragma unroll
        for(int v = 0; v < 16; v++)
            acc[tp][v] = 0.0f;
#pragma unroll 1
    for(int tile = split; tile < t.ntiles; tile += t.splits) {
        const int n = tile / t.tpi, in = tile - n * t.tpi, ty = in / t.nx, tx = in - ty * t.nx;
        const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void *)(t.x + n * ximg), 0, (unsigned)(ximg * 2), 0x00020000);
        const __amdgpu_buffer_rsrc_t ry = __builtin_amdgcn_make_buffer_rsrc((void *)(t.dy + n * yimg), 0, (unsigned)(yimg * 2), 0x00020000);
        const int ox = std::min(tx * TW, t.W - TW), oy = std::min(ty * TR, t.H - TR);
#pragma unroll 1
        for(int step = 0; step < TR / 2 * (TW / 8); step++) { // eight columns of two rows
            const int y = oy + step / (TW / 8) * 2 + hi, x0 = ox + step % (TW / 8) * 8;
            uint4_t keep; // pixels that no tile before had
#pragma unroll
            for(int i = 0; i < 4; i++) {
                const unsigned pair = (x0 + 2 * i >= tx * TW ? 0xffffu : 0u) | (x0 + 2 * i + 1 >= tx * TW ? 0xffff0000u : 0u);
                keep[i] = y >= ty * TR ? pair : 0u;
            }
            auto load = [&](__amdgpu_buffer_rsrc_t r, int yy, int xx, int ld, int ch, int channels) {
                const bool there = ch < channels && (unsigned)yy < (unsigned)t.H && (unsigned)xx < (unsigned)t.W;
                return (unsigned)__builtin_amdgcn_raw_buffer_load_b16(r, there ? (unsigned)(((yy * t.W + xx) * ld + ch) * 2) : OOB, 0, 0);
            };
            auto eight = [&](const unsigned *w) {
                uint4_t v;
#pragma unroll
                for(int i = 0; i < 4; i++)
                    v[i] = (w[2 * i] | w[2 * i + 1] << 16) & keep[i];
                return __builtin_bit_cast(half8_t, v);
            };
            unsigned g[8], p[3][10];
#pragma unroll
            for(int e = 0; e < 8; e++)
                g[e] = load(ry, y, x0 + e, t.ldy, k, t.K);
#pragma unroll
            for(int r = 0; r < 3; r++)
#pragma unroll
                for(int e = 0; e < 10; e++)
                    p[r][e] = load(rx, y + r - 1, x0 + e - 1, t.ldx, c, t.C);
#pragma unroll
            for(int tp = 0; tp < 9; tp++)
                acc[tp] = __builtin_amdgcn_mfma_f32_32x32x16_f16(eight(g), eight(p[tp / 3] + tp % 3), acc[tp], 0, 0, 0);
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // (the stores before)
#pragma unroll
    for(int tp = 0; tp < 9; tp++)
#pragma unroll
        for(int v = 0; v < 16; v++) {
            const float sum = acc[tp][v];
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, sum), ro,
                                                  c < t.C ? (unsigned)((((k0 + 8 * (v / 4) + 4 * hi + v % 4) * 9 + tp) * t.C + c) * 4) : OOB, 0, 0);
        }
}

// OVERLAP: tiles do not divide the image
template <int TW, int NST, bool OVERLAP> __global__ void __launch_bounds__(256, 1) conv_bwd_filter_strips(StripArgs t)
{
    using T = StripTile<TW, NST>;
    constexpr int TR = T::TR, SR = T::SR, NLX = T::NLX, NLY = T::NLY, XB = T::XB, YB = T::YB;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63, hi = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = wave >> 1, nt = wave & 1;
    const int b0 = xcd_remap(blockIdx.x, gridDim.x); // blocks of one share of the tiles are neighbours: they read the same pixels
    const int split = __builtin_amdgcn_readfirstlane(b0 / t.pairs), pair = b0 - split * t.pairs;
    const int kb = __builtin_amdgcn_readfirstlane(pair / t.pairs_c), k0 = kb * 64, c0 = (pair - kb * t.pairs_c) * 64;

    // This lane's loads: offsets from the tile's first pixel (x: from the one left of and above it), and one bit per load for
    // those that read zeros: always, in tiles at the left and at the right border, in tiles that overlap.  The bit becomes
    // the top bit of the offset, which no buffer reaches.
    unsigned roffx[NLX], roffy[NLY];
    unsigned xdead = 0, xleft = 0, xright = 0, ydead = 0, ycols = 0, yrows = 0;
    const int dup_cols = t.nx * TW - t.W, dup_rows = t.tpi / t.nx * TR - t.H;
#pragma unroll
    for(int q = 0; q < NLX; q++) {
        const int L = q * 256 + tid, slot = L >> 3, r = slot / SR, col = slot - r * SR;
        const int chunk = (L & 7) ^ (((col >> 1) & 1) << 2);
        roffx[q] = (unsigned)(((r * t.W + col) * t.ldx + chunk * 8) * 2);
        xdead |= slot >= (TR + 2) * SR || chunk * 8 >= t.C - c0 ? 1u << q : 0u;
        xleft |= col == 0 ? 1u << q : 0u;
        xright |= col == TW + 1 ? 1u << q : 0u;
    }
#pragma unroll
    for(int q = 0; q < NLY; q++) {
        const int L = q * 256 + tid, pix = L >> 3, r = pix / TW, col = pix - r * TW;
        const int chunk = (L & 7) ^ (((col >> 1) & 1) << 2);
        roffy[q] = (unsigned)(((r * t.W + col) * t.ldy + chunk * 8) * 2);
        ydead |= chunk * 8 >= t.K - k0 ? 1u << q : 0u;
        ycols |= col < dup_cols ? 1u << q : 0u;
        yrows |= r < dup_rows ? 1u << q : 0u;
    }
    const int64_t ximg = (int64_t)t.H * t.W * t.ldx * 2, yimg = (int64_t)t.H * t.W * t.ldy * 2;
    struct Tile {
        const char *x, *y;
        unsigned xbase, ybase, xkill, ykill;
    };
    auto place = [&](int tile) { // (behind the last tile: zeros, that the number of loads does not depend on it)
        Tile r;
        const bool real = tile < t.ntiles;
        const int tl = real ? tile : 0, n = __builtin_amdgcn_readfirstlane(tl / t.tpi), in = tl - n * t.tpi;
        const int ty = __builtin_amdgcn_readfirstlane(in / t.nx), tx = in - ty * t.nx;
        const int ox = tx * TW + TW <= t.W ? tx * TW : t.W - TW, oy = ty * TR + TR <= t.H ? ty * TR : t.H - TR;
        r.x = (const char *)t.x + n * ximg + c0 * 2;
        r.y = (const char *)t.dy + n * yimg + k0 * 2;
        r.xbase = (unsigned)(((oy - 1) * t.W + ox - 1) * t.ldx * 2); // (rows above the image: negative, no buffer reaches them)
        r.ybase = (unsigned)((oy * t.W + ox) * t.ldy * 2);
        r.xkill = xdead | (ox == 0 ? xleft : 0u) | (ox + TW == t.W ? xright : 0u);
        r.ykill = ydead | (ox < tx * TW ? ycols : 0u) | (oy < ty * TR ? yrows : 0u);
        if(!real)
            r.xkill = r.ykill = 0xffffffffu;
        return r;
    };
    const unsigned xrange = (unsigned)(ximg - c0 * 2), yrange = (unsigned)(yimg - k0 * 2);
    auto load_piece = [&](const Tile &r, int b, int p) {
        if(p < NLX) {
            const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void *)r.x, 0, xrange, 0x00020000);
            const unsigned at = roffx[p], off = (at + r.xbase) | ((r.xkill << (31 - p)) & 0x80000000u);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_ptr_t)(smem + b * XB + (p * 4 + wave) * 1024), 16, off, 0, 0, 0);
        } else {
            const int q = p - NLX;
            const __amdgpu_buffer_rsrc_t ry = __builtin_amdgcn_make_buffer_rsrc((void *)r.y, 0, yrange, 0x00020000);
            const unsigned at = roffy[q], off = (at + r.ybase) | ((r.ykill << (31 - q)) & 0x80000000u);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(ry, (lds_ptr_t)(smem + 2 * XB + b * YB + (q * 4 + wave) * 1024), 16, off, 0, 0, 0);
        }
    };

    // Operand addresses: a lane of a transposing read points at column fp (second half: fp + 4) of its row and four channels.
    const int fp = (lane & 15) >> 2, fc = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
    const unsigned lds0 = (unsigned)(uintptr_t)(lds_ptr_t)smem;
    const int gcol = TW == 16 ? 8 * grp : 0, grow = grp * T::GROUP_ROWS;
    unsigned xa[3], ya[2];
#pragma unroll
    for(int s = 0; s < 3; s++) {
        const int col = gcol + fp + s, c = nt * 32 + fc;
        xa[s] = lds0 + ((grow + hi) * SR + col) * 128 + (((c >> 3) ^ (((col >> 1) & 1) << 2)) << 4) + (c & 7) * 2;
    }
#pragma unroll
    for(int h = 0; h < 2; h++) {
        const int col = gcol + fp, k = h * 32 + fc;
        ya[h] = lds0 + 2 * XB + ((grow + hi) * TW + col) * 128 + (((k >> 3) ^ (((col >> 1) & 1) << 2)) << 4) + (k & 7) * 2;
    }

    float16_t acc[9][2];
#pragma unroll
    for(int tp = 0; tp < 9; tp++)
#pragma unroll
        for(int h = 0; h < 2; h++)
#pragma unroll
            for(int v = 0; v < 16; v++)
                acc[tp][h][v] = 0.0f;

    int tile = split, b = 0;
    {
        const Tile first = place(tile);
#pragma unroll
        for(int p = 0; p < NLX + NLY; p++)
            load_piece(first, 0, p);
    }
    for(; tile < t.ntiles; tile += t.splits) {
        // this tile has arrived (everybody's share: the barrier), and everybody is done with the other buffer
        asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
        const Tile next = place(tile + t.splits);
        unsigned xs[3], ys[2];
#pragma unroll
        for(int s = 0; s < 3; s++)
            xs[s] = xa[s] + b * XB;
#pragma unroll
        for(int h = 0; h < 2; h++)
            ys[h] = ya[h] + b * YB;
        half8_t even[3][3], odd[2][3], grad[2][2];
        // reads what instruction U is the first to use
        auto read_for = [&](auto U) {
            constexpr int j = U.value / 18, m = U.value % 18, s = m % 6 / 2;
            if constexpr(j < NST) {
                if constexpr(m < 2)
                    grad[j & 1][m] = read_pixels<j * 2 * TW * 128>(ys[m]);
                if constexpr(j == 0 && m < 6 && m % 2 == 0)
                    even[0][s] = read_pixels<0>(xs[s]);
                if constexpr(m >= 6 && m < 12 && m % 2 == 0)
                    odd[j & 1][s] = read_pixels<(2 * j + 1) * SR * 128>(xs[s]);
                if constexpr(m >= 12 && m % 2 == 0)
                    even[(j + 1) % 3][s] = read_pixels<(2 * j + 2) * SR * 128>(xs[s]);
            }
        };
        each<0, AHEAD>(read_for);
        each<0, 18 * NST>([&](auto I) {
            constexpr int u = I.value, j = u / 18, m = u % 18, s = m % 6 / 2, h = m % 2, row = m / 6;
            read_for(std::integral_constant<int, u + AHEAD>());
            half8_t &px = row == 0 ? even[j % 3][s] : (row == 1 ? odd[j & 1][s] : even[(j + 1) % 3][s]);
            half8_t &gr = grad[j & 1][h];
            if constexpr(first_uses(u, NST) > 0) {
                asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(2 * reads_behind(u, NST)) : "memory");
                asm volatile("" : "+v"(px), "+v"(gr));
            }
            // (of its own accord the compiler gives sums only the 256 accumulation registers, sixteen of these eighteen, and spills)
            if constexpr(row * 3 + s == 8)
                asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+v"(acc[8][h]) : "v"(gr), "v"(px));
            else
                acc[row * 3 + s][h] = __builtin_amdgcn_mfma_f32_32x32x16_f16(gr, px, acc[row * 3 + s][h], 0, 0, 0);
            if constexpr(u % 4 == 3 && u / 4 < NLX + NLY) {
                __builtin_amdgcn_sched_barrier(0);
                load_piece(next, b ^ 1, u / 4);
            }
            __builtin_amdgcn_sched_barrier(0);
        });
        b ^= 1;
    }
    // (loads into this block's LDS may still be on their way; and so may the products of the last instructions, of which the compiler
    // knows only its own)
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");

    // (a share's partial result is one buffer: rows and columns beyond the filter are outside)
    const unsigned sbytes = (unsigned)t.K * 9u * (unsigned)t.C * 4u;
    const __amdgpu_buffer_rsrc_t ro =
        __builtin_amdgcn_make_buffer_rsrc((void *)((char *)t.partial + (int64_t)split * sbytes), 0, sbytes, 0x00020000);
    const int c = c0 + nt * 32 + (lane & 31);
    // group g finishes half g of the output channels; the other half goes to the other group
    float4_t *const red = (float4_t *)smem;
    auto leave = [&](auto H) {
#pragma unroll
        for(int tp = 0; tp < 9; tp++)
#pragma unroll
            for(int v = 0; v < 4; v++)
                red[(wave * 36 + tp * 4 + v) * 64 + lane] = float4_t{acc[tp][H.value][4 * v], acc[tp][H.value][4 * v + 1],
                                                                     acc[tp][H.value][4 * v + 2], acc[tp][H.value][4 * v + 3]};
    };
    bool nan = false;
    auto finish = [&](auto H) {
        const int k = k0 + H.value * 32 + 4 * hi;
#pragma unroll
        for(int tp = 0; tp < 9; tp++)
#pragma unroll
            for(int v = 0; v < 4; v++) {
                const float4_t o = red[((wave ^ 2) * 36 + tp * 4 + v) * 64 + lane];
#pragma unroll
                for(int e = 0; e < 4; e++) {
                    const float sum = acc[tp][H.value][4 * v + e] + o[e];
                    if constexpr(OVERLAP)
                        nan |= sum != sum;
                    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, sum), ro,
                                                          c < t.C ? (unsigned)((((k + 8 * v + e) * 9 + tp) * t.C + c) * 4) : OOB, 0, 0);
                }
            }
    };
    if(grp == 0)
        leave(std::integral_constant<int, 1>());
    else
        leave(std::integral_constant<int, 0>());
    __syncthreads();
    if(grp == 0)
        finish(std::integral_constant<int, 0>());
    else
        finish(std::integral_constant<int, 1>());
    if constexpr(!OVERLAP)
        return;
    volatile int *const found = (volatile int *)smem;
    auto any = [&](bool here) { // (barriers that do not wait for the stores)
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        found[wave] = __builtin_amdgcn_ballot_w64(here) != 0;
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        return (found[0] | found[1] | found[2] | found[3]) != 0;
    };
    if(any(nan) && any(infinity_under_overlap<TW, TR>(t, split, c0)))
        strips_again<TW, TR>(t, split, k0 + grp * 32, c, ro); // (over what this wavefront has stored)
}

template <int TW, int NST, bool OVERLAP> int launch_as(const StripArgs &t, int blocks, hipStream_t st)
{
    constexpr int lds = StripTile<TW, NST>::LDS;
    const auto kern = conv_bwd_filter_strips<TW, NST, OVERLAP>;
    static const hipError_t allowed = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if(allowed != hipSuccess)
        return (int)allowed;
    kern<<<blocks, 256, lds, st>>>(t);
    SAGA_CHECK_LAUNCH();
    return 0;
}

template <int TW, int NST> int launch(const StripArgs &t, int blocks, hipStream_t st)
{
    return t.W % TW || t.H % StripTile<TW, NST>::TR ? launch_as<TW, NST, true>(t, blocks, st) : launch_as<TW, NST, false>(t, blocks, st);
}

int tile_rows(int tw, int nst) { return (tw == 16 ? 2 : 4) * nst; }

} // namespace

// Where a block walks three tiles or more, and where that takes less than tiles of a GEMM (conv_bwd_filter_dma).  Both launches, the
// first tile's way to LDS and the sum over partial results are 14 us, the partial results themselves (38 MB from 256 blocks of 64 x 64) up
// to 8, a tile of 16x16 3, the look for NaNs where tiles overlap 1.  What tiles have twice or channels that a block of 64 lacks cost as much as what counts, and more of
// it than the GEMM's tiles have.  us, GEMM / strips (before, whole rows in LDS for 64->64 with one operand per tap: 96 at 256x56x56):
//   64->64   256x56x56   121 /  67    64->64    64x56x56  45 / 34    64->64    32x56x56 (2 tiles) 31.4 / 30.7
//   64->64   16x256x256  170 /  82    16->16   256x56x56  66 / 48    64->64    16x56x56 (1 tile)  26.5 / 27.2
//   128->64  16x256x256  274 / 139    32->32    64x56x56  33 / 29    32->32   128x16x16 (1)       15.0 / 22.3
//   128->128 16x128x128  111 /  77    24->24  64x112x112  64 / 48    128->128  23x25x25 (2)       28.2 / 29.6
//   512->512 16x32x32    102 /  81    80->160   64x56x56 121 / 72    96->96     8x56x56 (2)       24.2 / 26.9
// and left to the GEMM for what tiles have twice or channels lack:
//   512->512 16x17x17     50 /  74    512->512   9x17x33  55 / 67    40->40   100x34x18           20 / 28
//   40->312  31x20x20     22 /  28    72->72    70x28x9   19 / 24    16->368   11x67x67           25 / 32
// (139 us for 155 GFLOP: 1240 TFLOP/s behind the fixed part, what a large matrix product reaches on this card.)
FilterStrips plan_filter_strips(const ConvGeom &g, int cus, double other_ns)
{
    FilterStrips best = {0, 0, 0, 0};
    if(g.R != 3 || g.S != 3 || g.stride != 1 || g.pad != 1 || g.dil != 1 || g.group != 1 || g.P != g.H || g.Q != g.W)
        return best;
    const int64_t pairs = (int64_t)((g.K + 63) / 64) * ((g.C + 63) / 64);
    if(pairs > 4 * cus || (int64_t)g.K * 9 * g.C * 4 >= 0x7fff0000ll)
        return best;
    const int share = std::max(1, cus / (int)pairs);
    int64_t least = 0;
    for(int tw : {16, 8})
        for(int nst : {8, 7}) {
            const int tr = tile_rows(tw, nst);
            if(g.W < tw || g.H < tr)
                continue;
            const int64_t tiles = (int64_t)((g.W + tw - 1) / tw) * ((g.H + tr - 1) / tr) * g.N;
            const int splits = (int)std::min<int64_t>(tiles, share);
            const int64_t each = (tiles + splits - 1) / splits, cost = each * (18 * nst + 16); // instructions, and a tile's own time
            if(tiles < 0x7fffffff && (!least || cost < least)) {
                least = cost;
                const double ns = 14000 + (g.W % tw || g.H % tr ? 1300 : 0) + 19.0 * cost + 0.8e-3 * splits * g.K * 9.0 * g.C;
                best = {tw, each >= 3 && ns < other_ns ? nst : 0, (int)pairs, splits};
            }
        }
    return best;
}

int launch_filter_strips(const FilterStrips &p, const half_t *x, int64_t ldx, const half_t *dy, int64_t ldy, float *partial,
                         const ConvGeom &g, hipStream_t st)
{
    const int64_t px = (int64_t)g.H * g.W;
    if(px * ldx * 2 >= 0x7fff0000ll || px * ldy * 2 >= 0x7fff0000ll)
        return SAGA_HIP_EUNSUPPORTED; // an image is one buffer
    const int tr = tile_rows(p.tw, p.nst);
    StripArgs t;
    t.x = x;
    t.dy = dy;
    t.partial = partial;
    t.ldx = (int)ldx;
    t.ldy = (int)ldy;
    t.H = g.H;
    t.W = g.W;
    t.C = g.C;
    t.K = g.K;
    t.nx = (g.W + p.tw - 1) / p.tw;
    t.tpi = t.nx * ((g.H + tr - 1) / tr);
    t.ntiles = t.tpi * g.N;
    t.pairs = p.pairs;
    t.pairs_c = (g.C + 63) / 64;
    t.splits = p.splits;
    const int blocks = p.pairs * p.splits;
    if(p.tw == 16)
        return p.nst == 8 ? launch<16, 8>(t, blocks, st) : launch<16, 7>(t, blocks, st);
    return p.nst == 8 ? launch<8, 8>(t, blocks, st) : launch<8, 7>(t, blocks, st);
}
