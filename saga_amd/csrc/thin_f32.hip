// fp32 convolutions of one to four input channels (grey values, colours) on the bf16 matrix unit (split_f32.hpp).
//
// The reduction is (channel, tap) in the filter's own order, in steps of sixteen.  A block keeps its channels' filter in LDS,
// in three parts and in the order of the lanes, and walks tiles of 256 or 512 output pixels, 64 to a wavefront: what they see of
// the padded images is a run of consecutive positions, which it loads once per channel, as it is, and from which a lane
// picks the eight numbers of its pixel for a step (the offsets come from a table) and splits them.
//
// The table kernel of stream_f32.hip and the tiles in LDS of conv_f32.hip, which did this before, load every tap of every
// pixel by itself.  us, launch included, before -> now: 7x7 3->64 at 8x224x224, stride 2  43 -> 30; 5x5 1->32 at 64x28x28
// 11.4 -> 7.0; at 512x28x28 33 -> 22; 3x3 3->16 at 128x32x32 11.2 -> 9.3; 3x3 4->130 at 16x64x64 34 -> 28.  The large ones wait for
// the picks from LDS (of a stride of two, from every other bank), the small ones for the launch and two trips to memory.
#include "split_f32.hpp"
#include "thin_f32.hpp"
#include "out_f32.hpp"

#include <algorithm>

namespace {

constexpr int MOST = 256;        // reduction indices
constexpr int LDS_ROOM = 150 * 1024;

struct ThinArgs {
    const float *x, *w;
    unsigned x_bytes, w_bytes;
    int batch, M, C, CRS, steps; // images, pixels, channels, reduction indices and steps
    int IH, IW, pad, stride, dil, R, S;
    int pitch, plane, window;    // of the padded images; positions of a tile
    int tiles, walkers, nblk_n;  // tiles of pixels, blocks that share them, blocks along the channels
    FastDiv ow, oh, by_pitch, by_plane;
    long long x_sn, x_sc, x_sh, x_sw;
    long long w_sn, w_sc, w_sr, w_ss;
    OutArgs o;
};

// POOL: a max pooling of 2x2 windows behind it (out_f32.hpp): a quarter of the results to store, and none to read again.  us, both launches / this:
// 5x5 1->32 at 64x28x28 15.1 / 8.7, at 512x28x28 43 / 25; 3x3 3->64 at 8x224x224 86 / 54.
template <int TN, int WAVES, bool EX, bool POOL> __global__ void __launch_bounds__(64 * WAVES, 2) stream_f32_k_thin(ThinArgs g)
{
    extern __shared__ __attribute__((aligned(16))) char lds[];
    __shared__ __attribute__((aligned(16))) int at_tap[MOST], w_at[MOST]; // of a reduction index: in the window; in the filter (bytes)
    __shared__ __attribute__((aligned(16))) float chan[2][32 * TN];
    constexpr int TM = 2, PIXELS = 64 * WAVES, THREADS = 64 * WAVES;
    const int tid = threadIdx.x, lane = tid & 63, fr = lane & 31, fk = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int walker = blockIdx.x / g.nblk_n, n0 = (blockIdx.x - walker * g.nblk_n) * 32 * TN;
    uint4_t *const parts = (uint4_t *)lds; // [32 channels][step][part][lane]
    float *const win = (float *)(lds + TN * g.steps * 3072);
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void *)g.x, 0, (int)g.x_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void *)g.w, 0, (int)g.w_bytes, 0x00020000);

    EpilogueF32::Raw raw;
    if(EX && g.o.e.affine() && tid < 32 * TN)
        raw = g.o.e.fetch(n0 + tid < g.o.N ? n0 + tid : g.o.N - 1);
    if(tid < g.steps * 16) {
        const int RS = g.R * g.S, c = tid / RS, tap = tid - c * RS, r = tap / g.S, s = tap - r * g.S;
        const bool in = tid < g.CRS;
        at_tap[tid] = in ? c * g.window + r * g.dil * g.pitch + s * g.dil : 0; // (behind the last the filter is zero)
        w_at[tid] = in ? (int)((c * g.w_sc + r * g.w_sr + s * g.w_ss) * 4) : -1;
    }
    auto place = [&](int m, int &n, int &oy, int &ox) { place_pixel<POOL>(g.ow, g.oh, m, n, oy, ox); };
    auto virt = [&](int n, int oy, int ox) { return n * g.plane + oy * g.stride * g.pitch + ox * g.stride; };
    auto load_window = [&](int tile) {
        int n, oy, ox;
        place(tile * PIXELS, n, oy, ox);
        const int lo = virt(n, oy, ox);
        for(int p0 = tid; p0 < g.window; p0 += 4 * THREADS) {
            unsigned off[4];
#pragma unroll
            for(int q = 0; q < 4; q++) {
                const int v = lo + p0 + THREADS * q, im = g.by_plane.div(v), rest = v - im * g.plane;
                const int row = g.by_pitch.div(rest), y = row - g.pad, x = rest - row * g.pitch - g.pad;
                const bool in = im < g.batch && (unsigned)y < (unsigned)g.IH && (unsigned)x < (unsigned)g.IW;
                off[q] = in ? (unsigned)((im * g.x_sn + y * g.x_sh + x * g.x_sw) * 4) : OUT_NOWHERE;
            }
            for(int c = 0; c < g.C; c++) {
                float f[4];
#pragma unroll
                for(int q = 0; q < 4; q++)
                    f[q] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rx, off[q], (unsigned)(c * g.x_sc * 4), 0));
#pragma unroll
                for(int q = 0; q < 4; q++)
                    if(p0 + THREADS * q < g.window)
                        win[c * g.window + p0 + THREADS * q] = f[q];
            }
        }
        return lo;
    };
    int lo = load_window(walker);
    __syncthreads();
    constexpr int AT_ONCE = WAVES == 8 && TN == 2 ? 4 : 1; // trips to memory of a long filter (of a short one there is one)
    for(int i0 = tid; i0 < TN * g.steps * 64; i0 += AT_ONCE * THREADS) {
        float v[AT_ONCE][8];
#pragma unroll
        for(int u = 0; u < AT_ONCE; u++) {
            const int i = i0 + u * THREADS, ln = i & 63, q = i >> 6, t = q >= g.steps, step = q - t * g.steps;
            const int n = n0 + 32 * t + (ln & 31);
            const bool in = q < TN * g.steps && n < g.o.N;
#pragma unroll
            for(int j = 0; j < 8; j++) {
                const int k = in ? w_at[step * 16 + 8 * (ln >> 5) + j] : -1;
                v[u][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                        rw, k >= 0 ? (unsigned)(n * g.w_sn * 4) + (unsigned)k : OUT_NOWHERE, 0, 0));
            }
        }
#pragma unroll
        for(int u = 0; u < AT_ONCE; u++) {
            const int i = i0 + u * THREADS, q = i >> 6;
            if(q >= TN * g.steps)
                break;
            Parts p;
            split3_any(v[u], p);
#pragma unroll
            for(int h = 0; h < 3; h++)
                parts[(q * 3 + h) * 64 + (i & 63)] = p.v[h];
        }
    }
    if(EX && g.o.e.affine() && tid < 32 * TN)
        g.o.e.leave(raw, chan[0][tid], chan[1][tid]);

    for(int tile = walker; tile < g.tiles; tile += g.walkers) {
        if(tile != walker) {
            __syncthreads();
            lo = load_window(tile);
        }
        __syncthreads();
        int at[TM], pn[TM], py[TM], px[TM];
        bool ok[TM];
#pragma unroll
        for(int i = 0; i < TM; i++) {
            const int m = tile * PIXELS + 64 * wave + 32 * i + fr;
            ok[i] = m < g.M;
            place(ok[i] ? m : tile * PIXELS, pn[i], py[i], px[i]);
            at[i] = virt(pn[i], py[i], px[i]) - lo;
        }
        float16_t acc[TM][TN], low[TM][TN];
#pragma unroll
        for(int i = 0; i < TM; i++)
#pragma unroll
            for(int t = 0; t < TN; t++)
#pragma unroll
                for(int v = 0; v < 16; v++)
                    acc[i][t][v] = low[i][t][v] = 0.0f;
        auto pick = [&](int step, float(&f)[TM][8]) {
            const int4 a = *(const int4 *)&at_tap[step * 16 + 8 * fk], b = *(const int4 *)&at_tap[step * 16 + 8 * fk + 4];
            const int o[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
            for(int i = 0; i < TM; i++)
#pragma unroll
                for(int j = 0; j < 8; j++)
                    f[i][j] = win[at[i] + o[j]];
        };
        for(int step = 0; step < g.steps; step++) {
            float f[TM][8];
            pick(step, f);
            uint4_t q[TN][3];
#pragma unroll
            for(int t = 0; t < TN; t++)
#pragma unroll
                for(int h = 0; h < 3; h++)
                    q[t][h] = parts[((t * g.steps + step) * 3 + h) * 64 + lane];
            Parts p[TM];
#pragma unroll
            for(int i = 0; i < TM; i++)
                split3(f[i], p[i]);
#pragma unroll
            for(int j = 0; j < SPLIT_PRODUCTS; j++)
#pragma unroll
                for(int i = 0; i < TM; i++)
#pragma unroll
                    for(int t = 0; t < TN; t++)
                        mfma_split(j, p[i], q[t], acc[i][t], low[i][t]);
        }
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
        if(__builtin_amdgcn_ballot_w64(bad != bad)) { // operands without three parts: in fp32 products
#pragma unroll
            for(int i = 0; i < TM; i++)
#pragma unroll
                for(int t = 0; t < TN; t++)
#pragma unroll
                    for(int v = 0; v < 16; v++)
                        acc[i][t][v] = 0.0f;
            for(int step = 0; step < g.steps; step++) {
                float f[TM][8];
                pick(step, f);
#pragma unroll
                for(int t = 0; t < TN; t++) {
                    uint4_t q[3];
#pragma unroll
                    for(int h = 0; h < 3; h++)
                        q[h] = parts[((t * g.steps + step) * 3 + h) * 64 + lane];
#pragma unroll
                    for(int j = 0; j < 8; j++) {
                        const bool in = step * 16 + 8 * fk + j < g.CRS; // (what a lane picks behind the last may be anything)
#pragma unroll
                        for(int i = 0; i < TM; i++)
                            acc[i][t] = __builtin_amdgcn_mfma_f32_32x32x2f32(joined(q, j), in ? f[i][j] : 0.0f, acc[i][t], 0, 0, 0);
                    }
                }
            }
        }
        const FourOut<EX, POOL> out(g.o, fk);
        int first = n0;
        asm volatile("" : "+s"(first)); // (or every value's scalar offset is kept from one tile to the next)
#pragma unroll
        for(int i = 0; i < TM; i++) {
            const unsigned op = out.out_at(ok[i], pn[i], py[i], px[i]), zp = out.z_at(ok[i], pn[i], py[i], px[i]);
#pragma unroll
            for(int t = 0; t < TN; t++) {
                Four was[4], res[4];
#pragma unroll
                for(int v = 0; v < 4; v++) {
                    was[v] = out.before(op, first + 32 * t + 8 * v);
                    res[v] = out.residual(zp, first + 32 * t + 8 * v);
                }
#pragma unroll
                for(int v = 0; v < 4; v++)
                    out.store(op, first + 32 * t + 8 * v, {acc[i][t][4 * v], acc[i][t][4 * v + 1], acc[i][t][4 * v + 2], acc[i][t][4 * v + 3]},
                              was[v], res[v], &chan[0][32 * t + 8 * v + 4 * fk], &chan[1][32 * t + 8 * v + 4 * fk]);
            }
        }
    }
}

template <int TN, int WAVES, bool EX, bool POOL = false> int launch(const ThinArgs &g, size_t bytes, hipStream_t st)
{
    auto kern = stream_f32_k_thin<TN, WAVES, EX, POOL>;
    static const hipError_t attr = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, LDS_ROOM);
    if(attr != hipSuccess)
        return (int)attr;
    kern<<<g.walkers * g.nblk_n, 64 * WAVES, bytes, st>>>(g);
    SAGA_CHECK_LAUNCH();
    return 0;
}

} // namespace

// what there is to launch: wavefronts of a block, channels of a block in 32s, its LDS
struct Launch {
    int waves, tn;
    long long bytes;
};

static int describe(const SagaTensorView *x, const SagaTensorView *w, const SagaTensorView *y, const ConvGeom &c, float alpha, float beta,
                    const StreamEpilogue &e, bool pool, ThinArgs &g, Launch &l)
{
    const long long xb = extent_of(x), wb = extent_of(w);
    if(c.C > 4 || c.group != 1 || (long long)c.C * c.R * c.S > MOST || xb < 0 || wb < 0 || xb > OUT_NOWHERE || wb > OUT_NOWHERE ||
       !describe_out(y, alpha, beta, e, g.o))
        return SAGA_HIP_EUNSUPPORTED;
    if(pool && (beta != 0.0f || e.z || c.P < 2 || c.Q < 2))
        return SAGA_HIP_EUNSUPPORTED;
    const int P = pool ? c.P / 2 : c.P, Q = pool ? c.Q / 2 : c.Q; // (of windows)
    const long long pixels = ((long long)c.N * P * Q) << (2 * pool), pitch = c.W + 2ll * c.pad, plane = pitch * (c.H + 2ll * c.pad);
    if(pixels >= 1ll << 30 || (c.N + 1) * plane >= 1ll << 30)
        return SAGA_HIP_EUNSUPPORTED;
    g.x = (const float *)x->ptr;
    g.w = (const float *)w->ptr;
    g.x_bytes = (unsigned)xb;
    g.w_bytes = (unsigned)wb;
    g.batch = c.N;
    g.M = (int)pixels;
    g.C = c.C;
    g.CRS = c.C * c.R * c.S;
    g.steps = (g.CRS + 15) / 16;
    g.IH = c.H; g.IW = c.W;
    g.pad = c.pad; g.stride = c.stride; g.dil = c.dil;
    g.R = c.R; g.S = c.S;
    g.pitch = (int)pitch;
    g.plane = (int)plane;
    // positions from the first pixel's first tap to the last one's last: rows skip what is right of the last pixel and stride - 1
    // rows, images what is below
    auto window_of = [&](long long count) {
        const long long taps = (c.R - 1ll) * c.dil * pitch + (c.S - 1ll) * c.dil + 1;
        if(pool) { // the same of windows of two rows and columns, the last one's last pixel a row below and a column beside its first
            const long long n = count / 4 - 1, rows = (n + Q - 1) / Q, images = (n + (long long)P * Q - 1) / ((long long)P * Q);
            return 2 * n * c.stride + rows * 2 * c.stride * (pitch - Q) + images * std::max(0ll, plane - 2ll * P * c.stride * pitch) +
                   c.stride * (pitch + 1) + taps;
        }
        const long long n = count - 1, rows = (n + c.Q - 1) / c.Q, images = (n + (long long)c.P * c.Q - 1) / ((long long)c.P * c.Q);
        const long long row = c.stride * (pitch - c.Q), image = plane - (long long)c.P * c.stride * pitch;
        return n * c.stride + rows * std::max(0ll, row) + images * std::max(0ll, image) + taps;
    };
    const int tn = g.o.N > 32 ? 2 : 1;
    auto bytes_of = [&](int waves) { return tn * g.steps * 3072ll + window_of(64 * waves) * c.C * 4; };
    // Eight wavefronts to a filter that takes a CU's LDS, or to rows so long that the tile's window is mostly above and below it
    int waves = tn * g.steps >= 8 || window_of(256) > 768 * c.stride * c.stride ? 8 : 4;
    if(waves == 8 && bytes_of(8) > LDS_ROOM)
        waves = 4;
    const long long bytes = bytes_of(waves);
    if(bytes > LDS_ROOM || (tn * g.steps >= 8 && pixels < 64 * 512)) // a long filter on a few CUs takes longer to split than to use
        return SAGA_HIP_EUNSUPPORTED;
    g.window = (int)window_of(64 * waves);
    g.tiles = (int)((pixels + 64 * waves - 1) / (64 * waves));
    g.nblk_n = (g.o.N + 32 * tn - 1) / (32 * tn);
    g.walkers = std::min(g.tiles, std::max(1, (bytes <= 75 * 1024 ? 512 : 256) / g.nblk_n));
    g.ow = fast_div(Q);
    g.oh = fast_div(P);
    g.by_pitch = fast_div(g.pitch);
    g.by_plane = fast_div(g.plane);
    g.x_sn = x->strides[0]; g.x_sc = x->strides[1]; g.x_sh = x->strides[2]; g.x_sw = x->strides[3];
    g.w_sn = w->strides[0]; g.w_sc = w->strides[1]; g.w_sr = w->strides[2]; g.w_ss = w->strides[3];
    l = {waves, tn, bytes};
    return 0;
}

bool thin_f32_maxpool_ok(const SagaTensorView *x, const SagaTensorView *w, const SagaTensorView *y, const ConvGeom &c)
{
    ThinArgs g = {};
    Launch l;
    return describe(x, w, y, c, 1.0f, 0.0f, StreamEpilogue(), true, g, l) == 0;
}

int thin_f32_conv(const SagaTensorView *x, const SagaTensorView *w, const SagaTensorView *y, const ConvGeom &c, float alpha,
                  float beta, const StreamEpilogue &e, hipStream_t st, bool pool)
{
    ThinArgs g = {};
    Launch l;
    const int r = describe(x, w, y, c, alpha, beta, e, pool, g, l);
    if(r)
        return r;
    const int waves = l.waves, tn = l.tn;
    const long long bytes = l.bytes;
    if(pool) {
        if(waves == 4)
            return tn == 1 ? launch<1, 4, true, true>(g, (size_t)bytes, st) : launch<2, 4, true, true>(g, (size_t)bytes, st);
        return tn == 1 ? launch<1, 8, true, true>(g, (size_t)bytes, st) : launch<2, 8, true, true>(g, (size_t)bytes, st);
    }
    const bool ex = beta != 0.0f || e.bias || e.bn_s || e.z || e.relu;
    if(waves == 4) {
        if(tn == 1)
            return ex ? launch<1, 4, true>(g, (size_t)bytes, st) : launch<1, 4, false>(g, (size_t)bytes, st);
        return ex ? launch<2, 4, true>(g, (size_t)bytes, st) : launch<2, 4, false>(g, (size_t)bytes, st);
    }
    if(tn == 1)
        return ex ? launch<1, 8, true>(g, (size_t)bytes, st) : launch<1, 8, false>(g, (size_t)bytes, st);
    return ex ? launch<2, 8, true>(g, (size_t)bytes, st) : launch<2, 8, false>(g, (size_t)bytes, st);
}
