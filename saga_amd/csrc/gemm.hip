// Row-major GEMM used by the fully-connected node: C = alpha*op(A)*op(B) + beta*C, either
// operand may be stored transposed.
//  * fp16: gemm_mfma_f16, 64x64x128 block tiles on v_mfma_f32_32x32x16_f16 (one 32x32 tile per
//    wave), operands staged through LDS with the reduction index contiguous; an operand
//    stored with the other index contiguous is transposed on its way into LDS; gemm_split_f16,
//    32x32 tiles whose reduction is split over a block, for grids that leave compute units idle.
//  * fp32: gemm_split_f32, 16x16 or 32x32 tiles whose reduction is split over a block, for small grids; stream_f32_gemm
//    (stream_f32.hip) for large ones; gemm_mfma_f32, 64x64x16 LDS tiles on v_mfma_f32_32x32x2_f32, for reductions
//    of up to 16 and operands beyond 2 GB.
#include "stream_f32.hpp"

namespace {

// fp32 on the matrix cores through LDS: one 32x32 tile per wavefront, 8 instructions per 16-deep slice.  A lane feeds A[m = lane%32][k = lane/32] and B[k][n = lane%32] and ends up with column
// n = lane%32, rows 8*(v/4) + 4*(lane/32) + v%4 of the tile.
__global__ void __launch_bounds__(256)
    gemm_mfma_f32(int tA, int tB, int M, int N, int K, float alpha, const float *__restrict__ A, int lda,
                  const float *__restrict__ B, int ldb, float beta, float *__restrict__ C, int ldc,
                  const float *__restrict__ bias, int relu)
{
    typedef float float16_t __attribute__((ext_vector_type(16)));
    constexpr int BM = 64, BN = 64, BK = 16;
    __shared__ float As[BK][BM + 4];
    __shared__ float Bs[BK][BN + 4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32;
    const int fr = lane & 31, fk = lane >> 5;
    float16_t acc;
#pragma unroll
    for(int v = 0; v < 16; v++)
        acc[v] = 0.0f;
    for(int k0 = 0; k0 < K; k0 += BK) {
        for(int e = tid; e < BM * BK; e += 256) {
            int mm, kk;
            if(tA) { mm = e % BM; kk = e / BM; } else { kk = e % BK; mm = e / BK; }
            const int gm = m0 + mm, gk = k0 + kk;
            float v = 0;
            if(gm < M && gk < K)
                v = tA ? A[(int64_t)gk * lda + gm] : A[(int64_t)gm * lda + gk];
            As[kk][mm] = v;
        }
        for(int e = tid; e < BN * BK; e += 256) {
            int nn, kk;
            if(tB) { kk = e % BK; nn = e / BK; } else { nn = e % BN; kk = e / BN; }
            const int gn = n0 + nn, gk = k0 + kk;
            float v = 0;
            if(gn < N && gk < K)
                v = tB ? B[(int64_t)gn * ldb + gk] : B[(int64_t)gk * ldb + gn];
            Bs[kk][nn] = v;
        }
        __syncthreads();
#pragma unroll
        for(int kk = 0; kk < BK / 2; kk++)
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(As[2 * kk + fk][wr + fr], Bs[2 * kk + fk][wc + fr], acc, 0, 0, 0);
        __syncthreads();
    }
    const int gn = n0 + wc + fr;
    if(gn >= N)
        return;
#pragma unroll
    for(int v = 0; v < 16; v++) {
        const int gm = m0 + wr + 8 * (v >> 2) + 4 * fk + (v & 3);
        if(gm >= M)
            continue;
        float *o = C + (int64_t)gm * ldc + gn;
        float r = alpha * acc[v];
        if(beta != 0.0f)
            r += beta * *o;
        if(bias)
            r += bias[gn];
        *o = relu && r == r ? fmaxf(r, 0.0f) : r;
    }
}

// what follows a product: a bias per column, in the product's type or fp32, and a relu; or the backward of a relu, whose output
// (of the product's type, its rows as far apart) is positive where the gradient passes.  Only the split reductions have the latter:
// of fc 64x10 -> 1024 it takes nothing (4.9 us with the launch), a launch of its own 4.6.
struct ColumnBias {
    const half_t *h;
    const float *f;
    int relu;
    const void *gate;
    template <typename T> __device__ __forceinline__ float pass(float v, int64_t at) const
    {
        // (the gradient in its own type first: one that overflows is infinite, and not a number where nothing passes)
        return gate ? (float)(T)v * ((float)((const T *)gate)[at] > 0.0f ? 1.0f : 0.0f) : v;
    }
    __device__ __forceinline__ float apply(float v, int n) const
    {
        if(h)
            v += (float)h[n];
        if(f)
            v += f[n];
        return relu && v == v ? fmaxf(v, 0.0f) : v;
    }
};

// One operand tile (64 rows x 32 reduction steps) from global memory into LDS rows of LDK
// halves.  kcontig: element (row, k) is at base[row*ld + k], else at base[k*ld + row].
// Every lane moves 8 elements that are contiguous in memory, with one 16-byte load when the
// run is in range and aligned.
// An iteration of the main loop takes GBK = 128 reduction steps (four 32-wide pieces per operand, eight 16-byte
// loads per lane in flight): with 32 the loop of a tall reduction (fc 2048 -> 1000 at batch 256: 64 blocks of 64
// iterations) paid one trip to memory per iteration and took 69 us; LDS rows are GLDK halves.
constexpr int GBK = 128;
constexpr int GLDK = GBK + 8;

__device__ __forceinline__ void gemm_stage(half_t (*dst)[GLDK], const half_t *__restrict__ base, int ld, bool kcontig,
                                           int row0, int rows, int k0, int K, bool vec_ok, int tid)
{
    half8_t v;
    if(kcontig) {
        const int r = tid >> 2, kk = (tid & 3) * 8;
        const int gr = row0 + r, gk = k0 + kk;
        const half_t *src = base + (int64_t)gr * ld + gk;
        if(vec_ok && gr < rows && gk + 8 <= K) {
            v = *(const half8_t *)src;
        } else {
#pragma unroll
            for(int j = 0; j < 8; j++)
                v[j] = (gr < rows && gk + j < K) ? src[j] : (half_t)0;
        }
        *(half8_t *)&dst[r][kk] = v;
    } else {
        const int kk = tid >> 3, r = (tid & 7) * 8;
        const int gr = row0 + r, gk = k0 + kk;
        const half_t *src = base + (int64_t)gk * ld + gr;
        if(vec_ok && gk < K && gr + 8 <= rows) {
            v = *(const half8_t *)src;
        } else {
#pragma unroll
            for(int j = 0; j < 8; j++)
                v[j] = (gk < K && gr + j < rows) ? src[j] : (half_t)0;
        }
#pragma unroll
        for(int j = 0; j < 8; j++)
            dst[r + j][kk] = v[j];
    }
}

__global__ void __launch_bounds__(256)
    gemm_mfma_f16(int tA, int tB, int M, int N, int K, float alpha, const half_t *__restrict__ A, int lda,
                  const half_t *__restrict__ B, int ldb, float beta, half_t *__restrict__ C, int ldc, int a_vec,
                  int b_vec, ColumnBias cb)
{
    __shared__ __attribute__((aligned(16))) half_t As[2][64][GLDK];
    __shared__ __attribute__((aligned(16))) half_t Bs[2][64][GLDK];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m0 = blockIdx.y * 64, n0 = blockIdx.x * 64;
    const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
    float16_t acc;
#pragma unroll
    for(int v = 0; v < 16; v++)
        acc[v] = 0.0f;
    const int frow = lane & 31, fk = (lane >> 5) * 8;
    const int KT = (K + GBK - 1) / GBK;
    // Vector path (both operands 16-byte loadable): all eight loads of an iteration are issued before the first
    // LDS write waits for one - branch-free, out-of-range runs read the operand's first bytes and are zeroed -
    // so an iteration pays one trip to memory, not eight.
    const bool fast = a_vec && b_vec;
    auto fetch = [&](const half_t *__restrict__ base, int ld, bool kcontig, int row0, int rows, int k0, bool &ok) {
        int gr, gk;
        if(kcontig) {
            gr = row0 + (tid >> 2); gk = k0 + (tid & 3) * 8;
            ok = gr < rows && gk + 8 <= K;
            return *(const half8_t *)(base + (ok ? (int64_t)gr * ld + gk : 0));
        }
        gk = k0 + (tid >> 3); gr = row0 + (tid & 7) * 8;
        ok = gk < K && gr + 8 <= rows;
        return *(const half8_t *)(base + (ok ? (int64_t)gk * ld + gr : 0));
    };
    auto put = [&](half_t(*dst)[GLDK], bool kcontig, half8_t v, bool ok) {
        if(!ok)
            v = half8_t{0, 0, 0, 0, 0, 0, 0, 0};
        if(kcontig) {
            *(half8_t *)&dst[tid >> 2][(tid & 3) * 8] = v;
        } else {
#pragma unroll
            for(int j = 0; j < 8; j++)
                dst[(tid & 7) * 8 + j][tid >> 3] = v[j];
        }
    };
    // a run that is only partly in range (K or the row count no multiple of 8) is rare: those tiles take the
    // element-wise path of gemm_stage
    auto partial = [&](int row0, int rows, int k0, bool kcontig) {
        return kcontig ? (K % 8 != 0 && k0 + GBK > K) : (rows % 8 != 0 && row0 + 64 > rows);
    };
    auto stage = [&](int buf, int k0) {
        if(fast && !partial(m0, M, k0, !tA) && !partial(n0, N, k0, tB)) {
            half8_t va[GBK / 32], vb[GBK / 32];
            bool oa[GBK / 32], ob[GBK / 32];
#pragma unroll
            for(int j = 0; j < GBK / 32; j++) {
                va[j] = fetch(A, lda, !tA, m0, M, k0 + 32 * j, oa[j]);
                vb[j] = fetch(B, ldb, tB, n0, N, k0 + 32 * j, ob[j]);
            }
#pragma unroll
            for(int j = 0; j < GBK / 32; j++) {
                put((half_t(*)[GLDK]) & As[buf][0][32 * j], !tA, va[j], oa[j]);
                put((half_t(*)[GLDK]) & Bs[buf][0][32 * j], tB, vb[j], ob[j]);
            }
            return;
        }
#pragma unroll
        for(int j = 0; j < GBK / 32; j++) {
            gemm_stage((half_t(*)[GLDK]) & As[buf][0][32 * j], A, lda, !tA, m0, M, k0 + 32 * j, K, a_vec, tid);
            gemm_stage((half_t(*)[GLDK]) & Bs[buf][0][32 * j], B, ldb, tB, n0, N, k0 + 32 * j, K, b_vec, tid);
        }
    };
    stage(0, 0);
    for(int kt = 0; kt < KT; kt++) {
        __syncthreads();
        const int cur = kt & 1;
        if(kt + 1 < KT)
            stage(cur ^ 1, (kt + 1) * GBK);
#pragma unroll
        for(int kk = 0; kk < GBK / 16; kk++) {
            const half8_t fa = *(const half8_t *)&As[cur][wm + frow][kk * 16 + fk];
            const half8_t fb = *(const half8_t *)&Bs[cur][wn + frow][kk * 16 + fk];
            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa, fb, acc, 0, 0, 0);
        }
    }
    const int n = n0 + wn + (lane & 31);
    if(n >= N)
        return;
#pragma unroll
    for(int v = 0; v < 16; v++) {
        const int m = m0 + wm + (v >> 2) * 8 + (lane >> 5) * 4 + (v & 3);
        if(m >= M)
            continue;
        half_t *o = C + (int64_t)m * ldc + n;
        const float r = alpha * acc[v];
        *o = (half_t)cb.apply(beta != 0.0f ? r + beta * (float)*o : r, n);
    }
}

// A lane of the kernels below loads N consecutive elements, at any address.  Where the operand ends before the run does, the run is moved
// to end there: every load is whole, whatever the sizes, without a branch, and the elements are put where they belong afterwards (rows
// that two lanes have got are written twice).  Nothing beyond the operand is read.  Loaded element by element where a dimension was no multiple of
// the run or an address not its own, all of them had to be there before the next could go out; us, before -> now, fp32 / fp16: 64x10x1024
// 7.9 -> 4.7 / 14 -> 4.7, 33x257x999 9.1 -> 5.0 / 19 -> 5.4, 23x1000x2041 15 -> 6.5 / 21 -> 7.3; the launch is 4.7.
typedef unsigned run_t __attribute__((ext_vector_type(4)));
typedef half_t any8_t __attribute__((ext_vector_type(8), aligned(2)));
typedef float any4_t __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ int run_of_rows(int n, int row, int rows) { return row < rows - n ? row : rows - n; }
__device__ __forceinline__ int64_t run_at(bool kcontig, int n, int ld, int row, int rows, int k, int K)
{
    return kcontig ? (int64_t)(row < rows ? row : rows - 1) * ld + run_of_rows(n, k, K)
                   : (int64_t)(k < K ? k : K - 1) * ld + run_of_rows(n, row, rows);
}
// steps k to k + N - 1, of which those beyond the reduction are zeros, from the run that was loaded for them
template <int N, typename V> __device__ __forceinline__ V run_of_steps(V v, int k, int K)
{
    run_t w = __builtin_bit_cast(run_t, v);
    const int by = k - run_of_rows(N, k, K);
    if(K % N) { // (or it is a whole run, or none)
        const unsigned far = N == 8 ? by & 4 : by & 2, near = N == 8 ? by & 2 : by & 1;
        w = far ? run_t{w[2], w[3], 0, 0} : w;
        w = near ? run_t{w[1], w[2], w[3], 0} : w;
        if(N == 8)
            w = by & 1 ? run_t{w[0] >> 16 | w[1] << 16, w[1] >> 16 | w[2] << 16, w[2] >> 16 | w[3] << 16, w[3] >> 16} : w;
    }
    return __builtin_bit_cast(V, by < N ? w : run_t{0, 0, 0, 0});
}

// The same for grids that leave compute units idle (few rows, or few outputs): a 32x32 tile per block of 8 wavefronts that
// split the reduction, every eighth slice of 64 steps each, and add their tiles through LDS in a fixed order.  What bounds
// such a product is the chain of trips to memory of one block: with 64x64 tiles fc 2048 -> 1000 ran in 16 blocks of 16
// dependent slices (1 sample: 34 -> 5 us, 256 samples: 31 -> 6 us).
// A slice is one cache line per row.  A wavefront fetches it in the order of memory (8 lanes per line), turns it through an
// LDS area of its own into operand order, and has the next slice in flight meanwhile; nothing is shared before the sum, so
// the loop holds no barrier.
constexpr int GS_K = 64, GS_LD = GS_K + 8, GS_WAVES = 8;

template <bool tA, bool tB, bool RUNS>
__global__ void __launch_bounds__(64 * GS_WAVES)
    gemm_split_f16(int M, int N, int K, float alpha, const half_t *__restrict__ A, int lda,
                   const half_t *__restrict__ B, int ldb, float beta, half_t *__restrict__ C, int ldc, ColumnBias cb)
{
    __shared__ __attribute__((aligned(16))) half_t st[GS_WAVES][2][32][GS_LD];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m0 = blockIdx.y * 32, n0 = blockIdx.x * 32;
    float16_t acc;
#pragma unroll
    for(int v = 0; v < 16; v++)
        acc[v] = 0.0f;
    // 8 consecutive elements in memory order: along the reduction (kcontig), or along the rows
    auto fetch = [&](half8_t(&d)[4], const half_t *__restrict__ base, int ld, bool kcontig, int row0, int rows, int k0) {
#pragma unroll
        for(int j = 0; j < 4; j++) {
            const int r = row0 + (kcontig ? (lane >> 3) + 8 * j : (lane & 3) * 8), k = k0 + (kcontig ? (lane & 7) * 8 : (lane >> 2) + 16 * j);
            if constexpr(RUNS) {
                d[j] = *(const any8_t *)(base + run_at(kcontig, 8, ld, r, rows, k, K));
            } else {
#pragma unroll
                for(int e = 0; e < 8; e++) {
                    const int re = kcontig ? r : r + e, ke = kcontig ? k + e : k;
                    const bool ok = re < rows && ke < K;
                    const half_t v = base[ok ? kcontig ? (int64_t)re * ld + ke : (int64_t)ke * ld + re : 0];
                    d[j][e] = ok ? v : (half_t)0;
                }
            }
        }
    };
    // (steps beyond the reduction become zeros here, not where they are loaded: that would wait for the load; rows beyond
    // the operand feed outputs that are not stored)
    auto put = [&](half_t(*d)[GS_LD], half8_t(&v)[4], bool kcontig, int row0, int rows, int k0) {
#pragma unroll
        for(int j = 0; j < 4; j++) {
            const int k = k0 + (kcontig ? (lane & 7) * 8 : (lane >> 2) + 16 * j);
            if(kcontig) {
                if(RUNS && k0 + GS_K > K)
                    v[j] = run_of_steps<8>(v[j], k, K);
                *(half8_t *)&d[(lane >> 3) + 8 * j][(lane & 7) * 8] = v[j];
            } else {
                if(k >= K)
                    v[j] = half8_t{0, 0, 0, 0, 0, 0, 0, 0};
                half_t(*const to)[GS_LD] = d + (lane & 3) * 8;
                const int col = (lane >> 2) + 16 * j;
                if(!RUNS || row0 + 32 <= rows || rows % 8 == 0) { // (no run was moved, or only whole ones behind the last row)
#pragma unroll
                    for(int e = 0; e < 8; e++)
                        to[e][col] = v[j][e];
                } else {
                    const int r = run_of_rows(8, row0 + (lane & 3) * 8, rows) - row0;
#pragma unroll
                    for(int e = 0; e < 8; e++)
                        if(r + e >= 0)
                            d[r + e][col] = v[j][e];
                }
            }
        }
    };
    const int slices = (K + GS_K - 1) / GS_K;
    const int fr = lane & 31, fk = (lane >> 5) * 8;
    half8_t va[4], vb[4];
    auto load = [&](int s) {
        fetch(va, A, lda, !tA, m0, M, s * GS_K);
        fetch(vb, B, ldb, tB, n0, N, s * GS_K);
    };
    if(wave < slices)
        load(wave);
    for(int s = wave; s < slices; s += GS_WAVES) {
        put(st[wave][0], va, !tA, m0, M, s * GS_K);
        put(st[wave][1], vb, tB, n0, N, s * GS_K);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if(s + GS_WAVES < slices)
            load(s + GS_WAVES);
#pragma unroll
        for(int kk = 0; kk < GS_K / 16; kk++) {
            const half8_t fa = *(const half8_t *)&st[wave][0][fr][kk * 16 + fk];
            const half8_t fb = *(const half8_t *)&st[wave][1][fr][kk * 16 + fk];
            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa, fb, acc, 0, 0, 0);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    float(*red)[32][33] = (float(*)[32][33]) & st[0][0][0][0];
    static_assert(sizeof(st) >= GS_WAVES * 32 * 33 * sizeof(float), "the tiles of the sum fit the staging area");
#pragma unroll
    for(int v = 0; v < 16; v++)
        red[wave][(v >> 2) * 8 + (lane >> 5) * 4 + (v & 3)][lane & 31] = acc[v];
    __syncthreads();
    const int n = n0 + (tid & 31);
#pragma unroll
    for(int h = 0; h < 2; h++) {
        const int ml = (tid >> 5) + 16 * h, m = m0 + ml;
        float r = 0;
#pragma unroll
        for(int w = 0; w < GS_WAVES; w++)
            r += red[w][ml][tid & 31];
        if(m < M && n < N) {
            half_t *o = C + (int64_t)m * ldc + n;
            r *= alpha;
            *o = (half_t)cb.pass<half_t>(cb.apply(beta != 0.0f ? r + beta * (float)*o : r, n), (int64_t)m * ldc + n);
        }
    }
}

} // namespace

// fp32, the same plan: T x T tiles (v_mfma_f32_16x16x4 / 32x32x2), W wavefronts that split the reduction in slices of 32
// steps (a cache line per row), DEPTH slices of each wavefront in flight.  Small grids are bound by the few compute units
// that work, and the streaming kernel there by the address unit besides, since its lanes load from a row each: fc 64x3136 ->
// 1024 ran in 64 blocks, 21 us; in 256 of 16x16 tiles it takes 10.
template <int T, int W, bool tA, bool tB, bool RUNS>
__global__ void __launch_bounds__(64 * W)
    gemm_split_f32(int M, int N, int K, float alpha, const float *__restrict__ A, int lda, const float *__restrict__ B, int ldb,
                   float beta, float *__restrict__ C, int ldc, ColumnBias cb)
{
    constexpr int KS = 32, LD = KS + 4, NL = T / 8, DEPTH = 2, NV = T * T / 64;
    typedef float acc_t __attribute__((ext_vector_type(NV)));
    __shared__ __attribute__((aligned(16))) float st[W][2][T][LD];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m0 = blockIdx.y * T, n0 = blockIdx.x * T;
    acc_t acc;
#pragma unroll
    for(int v = 0; v < NV; v++)
        acc[v] = 0.0f;
    constexpr int RL = T / 4, KL = 64 / RL; // lanes along the rows and steps per load, where the rows are contiguous
    auto fetch = [&](float4_t(&d)[NL], const float *__restrict__ base, int ld, bool kcontig, int row0, int rows, int k0) {
#pragma unroll
        for(int j = 0; j < NL; j++) {
            const int r = row0 + (kcontig ? (lane >> 3) + 8 * j : (lane % RL) * 4), k = k0 + (kcontig ? (lane & 7) * 4 : lane / RL + KL * j);
            if constexpr(RUNS) {
                d[j] = *(const any4_t *)(base + run_at(kcontig, 4, ld, r, rows, k, K));
            } else {
#pragma unroll
                for(int e = 0; e < 4; e++) {
                    const int re = kcontig ? r : r + e, ke = kcontig ? k + e : k;
                    const bool ok = re < rows && ke < K;
                    const float v = base[ok ? kcontig ? (int64_t)re * ld + ke : (int64_t)ke * ld + re : 0];
                    d[j][e] = ok ? v : 0.0f;
                }
            }
        }
    };
    // (steps beyond the reduction become zeros here, not where they are loaded: that would wait for the load)
    auto put = [&](float(*d)[LD], float4_t(&v)[NL], bool kcontig, int row0, int rows, int k0) {
#pragma unroll
        for(int j = 0; j < NL; j++) {
            const int k = k0 + (kcontig ? (lane & 7) * 4 : lane / RL + KL * j);
            if(kcontig) {
                if(RUNS && k0 + KS > K)
                    v[j] = run_of_steps<4>(v[j], k, K);
                *(float4_t *)&d[(lane >> 3) + 8 * j][(lane & 7) * 4] = v[j];
            } else {
                if(k >= K)
                    v[j] = float4_t{0, 0, 0, 0};
                float(*const to)[LD] = d + (lane % RL) * 4;
                const int col = lane / RL + KL * j;
                if(!RUNS || row0 + T <= rows || rows % 4 == 0) { // (no run was moved, or only whole ones behind the last row)
#pragma unroll
                    for(int e = 0; e < 4; e++)
                        to[e][col] = v[j][e];
                } else {
                    const int r = run_of_rows(4, row0 + (lane % RL) * 4, rows) - row0;
#pragma unroll
                    for(int e = 0; e < 4; e++)
                        if(r + e >= 0)
                            d[r + e][col] = v[j][e];
                }
            }
        }
    };
    const int slices = (K + KS - 1) / KS;
    const int fr = lane % T, fk = lane / T;
    float4_t va[DEPTH][NL], vb[DEPTH][NL];
    auto load = [&](int u, int s) {
        if(s >= slices)
            return;
        fetch(va[u], A, lda, !tA, m0, M, s * KS);
        fetch(vb[u], B, ldb, tB, n0, N, s * KS);
    };
#pragma unroll
    for(int u = 0; u < DEPTH; u++)
        load(u, wave + W * u);
    for(int s0 = wave; s0 < slices; s0 += W * DEPTH) {
#pragma unroll
        for(int u = 0; u < DEPTH; u++) {
            const int s = s0 + W * u;
            if(s >= slices)
                break;
            put(st[wave][0], va[u], !tA, m0, M, s * KS);
            put(st[wave][1], vb[u], tB, n0, N, s * KS);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            load(u, s + W * DEPTH);
            constexpr int STEP = 4 * (64 / T); // steps that one 16-byte read per lane covers
#pragma unroll
            for(int kk = 0; kk < KS; kk += STEP) {
                const float4_t fa = *(const float4_t *)&st[wave][0][fr][kk + 4 * fk];
                const float4_t fb = *(const float4_t *)&st[wave][1][fr][kk + 4 * fk];
#pragma unroll
                for(int e = 0; e < 4; e++) {
                    if constexpr(T == 32)
                        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[e], fb[e], acc, 0, 0, 0);
                    else
                        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[e], fb[e], acc, 0, 0, 0);
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
    }
    __syncthreads();
    float(*red)[T][T + 1] = (float(*)[T][T + 1]) & st[0][0][0][0];
    static_assert(sizeof(st) >= W * T * (T + 1) * sizeof(float), "the tiles of the sum fit the staging area");
#pragma unroll
    for(int v = 0; v < NV; v++) // column lane % T; rows: eights of fours (32x32), fours (16x16)
        red[wave][T == 32 ? (v >> 2) * 8 + fk * 4 + (v & 3) : fk * 4 + v][fr] = acc[v];
    __syncthreads();
    for(int e = tid; e < T * T; e += 64 * W) {
        const int ml = e / T, nl = e % T, m = m0 + ml, n = n0 + nl;
        float r = 0;
#pragma unroll
        for(int w = 0; w < W; w++)
            r += red[w][ml][nl];
        if(m < M && n < N) {
            float *o = C + (int64_t)m * ldc + n;
            r *= alpha;
            *o = cb.pass<float>(cb.apply(beta != 0.0f ? r + beta * *o : r, n), (int64_t)m * ldc + n);
        }
    }
}

template <int T, int W>
static void launch_split_f32(bool tA, bool tB, int M, int N, int K, float alpha, const float *A, int lda, const float *B, int ldb, float beta,
                             float *C, int ldc, const ColumnBias &cb, hipStream_t st)
{
    // (what is shorter than a run goes element by element)
    const bool runs = (tA ? M : K) >= 4 && (tB ? K : N) >= 4;
    auto kern = tA ? tB ? runs ? gemm_split_f32<T, W, true, true, true> : gemm_split_f32<T, W, true, true, false>
                        : runs ? gemm_split_f32<T, W, true, false, true> : gemm_split_f32<T, W, true, false, false>
                   : tB ? runs ? gemm_split_f32<T, W, false, true, true> : gemm_split_f32<T, W, false, true, false>
                        : runs ? gemm_split_f32<T, W, false, false, true> : gemm_split_f32<T, W, false, false, false>;
    kern<<<dim3((N + T - 1) / T, (M + T - 1) / T), 64 * W, 0, st>>>(M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, cb);
}

// Below one 64x64 tile per compute unit the reduction of a product in fp16 is split, unless it is shorter than there are tiles: then a tile's
// chain is short beside the work of the others (1024x1024: K = 1024 19 -> 14 us, 256 equal, 64 5.0 -> 5.4 us;
// 1000x2048, 512 tiles, K = 256: 12 -> 14 us).  A reduction of up to 16 is one slice in both, and loaded in runs there
// (64x1024, K = 10 6.3 -> 4.8 us, 600x300, K = 12 6.6 -> 4.8; 1000x512, K = 16 equal).
// In fp32 it is split up to one 32x32 tile per compute unit.
static bool splits(int M, int N, int K, int dtype)
{
    const int64_t t64 = ((int64_t)(M + 63) / 64) * ((N + 63) / 64), t32 = ((int64_t)(M + 31) / 32) * ((N + 31) / 32);
    return dtype == SAGA_HALF ? t64 <= 256 && (t64 <= 64 || K > t64) : t32 <= 256;
}

static int gemm(int transA, int transB, int M, int N, int K, float alpha, const void *A, int lda, const void *B, int ldb,
                float beta, void *C, int ldc, int dtype, const ColumnBias &cb, saga_stream_t stream)
{
    if(!A || !B || !C || M < 1 || N < 1 || K < 1)
        return SAGA_HIP_EINVAL;
    if(lda < (transA ? M : K) || ldb < (transB ? K : N) || ldc < N)
        return SAGA_HIP_ESHAPE;
    dim3 grid((N + 63) / 64, (M + 63) / 64);
    hipStream_t st = as_stream(stream);
    if(dtype == SAGA_HALF) {
        const int a_vec = lda % 8 == 0 && ((uintptr_t)A & 15) == 0, b_vec = ldb % 8 == 0 && ((uintptr_t)B & 15) == 0;
        if(splits(M, N, K, dtype)) {
            // (what is shorter than a run goes element by element)
            const bool runs = (transA ? M : K) >= 8 && (transB ? K : N) >= 8;
            auto kern = transA ? transB ? runs ? gemm_split_f16<true, true, true> : gemm_split_f16<true, true, false>
                                        : runs ? gemm_split_f16<true, false, true> : gemm_split_f16<true, false, false>
                               : transB ? runs ? gemm_split_f16<false, true, true> : gemm_split_f16<false, true, false>
                                        : runs ? gemm_split_f16<false, false, true> : gemm_split_f16<false, false, false>;
            kern<<<dim3((N + 31) / 32, (M + 31) / 32), 64 * GS_WAVES, 0, st>>>(M, N, K, alpha, (const half_t *)A, lda, (const half_t *)B,
                                                                             ldb, beta, (half_t *)C, ldc, cb);
            SAGA_CHECK_LAUNCH();
            return 0;
        }
        if(cb.gate)
            return SAGA_HIP_EUNSUPPORTED;
        gemm_mfma_f16<<<grid, 256, 0, st>>>(transA, transB, M, N, K, alpha, (const half_t *)A, lda, (const half_t *)B,
                                            ldb, beta, (half_t *)C, ldc, a_vec, b_vec, cb);
    } else if(dtype == SAGA_FLOAT) {
        // (one slice of the LDS tiles holds such a reduction)
        // us, stream / 16x16 tiles on 16 and on 4
        // wavefronts / 32x32 on 8: 64x1024x3136 21 / 11 / 13 / 23, 64x10x1024, by elements, 11 / 8 / 10 / 18, 64x3136x1024 13 / 12 / 10 / 9,
        // 128x1000x2048 16 / 18 / 15 / 17, 512x512x512 8.1 / 9.4 / 7.4 / 6.6, 300x300x32 4.7 / 3.6 / 2.7 / 3.4; beyond it
        // 512x1024x3136 43 / 69 / 57 / 46, 1024x1024x256 11 / 22 / 13 / 14).
        const int64_t t32 = ((int64_t)(M + 31) / 32) * ((N + 31) / 32), t16 = ((int64_t)(M + 15) / 16) * ((N + 15) / 16);
        if(splits(M, N, K, dtype)) {
            auto go = t16 <= 256 && K > 128   ? launch_split_f32<16, 16>
                      : t32 >= 192 && K > 64 ? launch_split_f32<32, 8>
                                             : launch_split_f32<16, 4>;
            go(transA, transB, M, N, K, alpha, (const float *)A, lda, (const float *)B, ldb, beta, (float *)C, ldc, cb, st);
            SAGA_CHECK_LAUNCH();
            return 0;
        }
        if(cb.gate)
            return SAGA_HIP_EUNSUPPORTED;
        if(K > 16) {
            const int r = stream_f32_gemm(transA, transB, M, N, K, alpha, (const float *)A, lda, (const float *)B, ldb, beta,
                                          (float *)C, ldc, cb.f, cb.relu, st);
            if(r != SAGA_HIP_EUNSUPPORTED)
                return r;
        }
        gemm_mfma_f32<<<grid, 256, 0, st>>>(transA, transB, M, N, K, alpha, (const float *)A, lda, (const float *)B, ldb,
                                            beta, (float *)C, ldc, cb.f, cb.relu);
    } else
        return SAGA_HIP_EUNSUPPORTED;
    SAGA_CHECK_LAUNCH();
    return 0;
}

extern "C" int saga_hip_gemm(int transA, int transB, int M, int N, int K, float alpha, const void *A, int lda,
                             const void *B, int ldb, float beta, void *C, int ldc, int dtype, saga_stream_t stream)
{
    return gemm(transA, transB, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, dtype, ColumnBias{nullptr, nullptr, 0, nullptr}, stream);
}

extern "C" int saga_hip_gemm_bias(int transA, int transB, int M, int N, int K, float alpha, const void *A, int lda,
                                  const void *B, int ldb, float beta, void *C, int ldc, int dtype, const void *bias, int bias_dtype,
                                  int relu, saga_stream_t stream)
{
    if(bias && bias_dtype != SAGA_FLOAT && !(bias_dtype == SAGA_HALF && dtype == SAGA_HALF))
        return SAGA_HIP_EUNSUPPORTED;
    const ColumnBias cb = {bias_dtype == SAGA_HALF ? (const half_t *)bias : nullptr, bias_dtype == SAGA_FLOAT ? (const float *)bias : nullptr,
                           relu, nullptr};
    return gemm(transA, transB, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, dtype, cb, stream);
}

extern "C" int saga_hip_gemm_relu_bwd_ok(int M, int N, int K, int dtype)
{
    return M > 0 && N > 0 && K > 0 && (dtype == SAGA_HALF || dtype == SAGA_FLOAT) && splits(M, N, K, dtype);
}

extern "C" int saga_hip_gemm_relu_bwd(int transA, int transB, int M, int N, int K, float alpha, const void *A, int lda, const void *B,
                                      int ldb, void *C, int ldc, int dtype, const void *y, saga_stream_t stream)
{
    if(!y)
        return SAGA_HIP_EINVAL;
    return gemm(transA, transB, M, N, K, alpha, A, lda, B, ldb, 0.0f, C, ldc, dtype, ColumnBias{nullptr, nullptr, 0, y}, stream);
}
