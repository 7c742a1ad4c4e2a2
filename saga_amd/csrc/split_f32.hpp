// fp32 products on the bf16 matrix unit: every operand as the sum of three bf16 numbers.
//
// A bf16 holds eight bits of an fp32's 24, so three hold all of them (h = bf16(x), m = bf16(x - h), l = bf16(x - h - m),
// both differences exact), and of the nine products of two such sums the six largest leave out less than 2^-24 of a
// product.  The bf16 instructions run at sixteen times the rate of the fp32 ones, so six of them take 3/8 of the time.
// The products of the leading parts and the smaller ones are added up apart, and together at the end: the small ones are
// not rounded to the large sum's last place one after another.  Against 64 bits (standard normal x N(0, 0.02), relative
// 2-norm of 1024 results): reduction of 64 4.6e-8 (fp32 instructions 1.6e-7), of 576 1.4e-7 (4.3e-7), of 4608 4.2e-7
// (1.2e-6); positive operands and operands over ten decades alike.
//
// The range of the operands: a bf16 has no bits below 2^-133, so that the parts of a number below 2^-110 would lose some.  What is
// split is therefore 2^24 times the number (fp32 numbers, the subnormal ones too, are multiples of 2^-149, their parts then of
// 2^-125, the last place of the smallest normal bf16), and a sum is brought back by 2^-48.  At the other end that makes
// numbers of 2^104 and sums of 2^80 infinite here.  They, infinities and NaNs leave a sum that is not finite, and a kernel that
// finds one takes it again in fp32 products.
#pragma once
#include "common.hpp"

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float float2_t __attribute__((ext_vector_type(2)));
typedef unsigned uint4_t __attribute__((ext_vector_type(4)));

struct Parts {
    uint4_t v[3];
};

template <typename V> __device__ __forceinline__ bf16x8_t part(V v) { return __builtin_bit_cast(bf16x8_t, v); }

__device__ __forceinline__ unsigned bf16_pair(float a, float b)
{
    const float2_t v = {a, b};
    return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2_t));
}

constexpr float SPLIT_UP = 0x1p24f, SPLIT_DOWN = 0x1p-24f, SPLIT_SUM = 0x1p-48f; // of an operand, of its parts, of a sum of products

// the three parts of eight numbers, the matrix instruction's operand of one lane each
__device__ __forceinline__ void split3(const float *x, Parts &p)
{
#pragma unroll
    for(int j = 0; j < 4; j++) {
        float a = x[2 * j] * SPLIT_UP, b = x[2 * j + 1] * SPLIT_UP;
        const unsigned h = bf16_pair(a, b);
        a -= __builtin_bit_cast(float, h << 16);
        b -= __builtin_bit_cast(float, h & 0xffff0000u);
        const unsigned m = bf16_pair(a, b);
        a -= __builtin_bit_cast(float, m << 16);
        b -= __builtin_bit_cast(float, m & 0xffff0000u);
        p.v[0][j] = h;
        p.v[1][j] = m;
        p.v[2][j] = bf16_pair(a, b);
    }
}

// The same for numbers that joined() gets back, of any kind: of one that has no parts the first is an infinity, the others
// are the halves of its bits.
__device__ __forceinline__ void split3_any(const float *x, Parts &p)
{
#pragma unroll
    for(int j = 0; j < 4; j++) {
        unsigned w[3] = {};
#pragma unroll
        for(int e = 0; e < 2; e++) {
            float r = x[2 * j + e] * SPLIT_UP;
            unsigned v[3];
#pragma unroll
            for(int i = 0; i < 3; i++) {
                v[i] = bf16_pair(r, r) & 0xffffu;
                r -= __builtin_bit_cast(float, v[i] << 16);
            }
            if((v[0] & 0x7f80u) == 0x7f80u) {
                const unsigned bits = __builtin_bit_cast(unsigned, x[2 * j + e]);
                v[0] = 0x7f80u;
                v[1] = bits & 0xffffu;
                v[2] = bits >> 16;
            }
#pragma unroll
            for(int i = 0; i < 3; i++)
                w[i] |= v[i] << 16 * e;
        }
#pragma unroll
        for(int i = 0; i < 3; i++)
            p.v[i][j] = w[i];
    }
}

// number j of eight that split3_any has split
template <typename V> __device__ __forceinline__ float joined(const V (&q)[3], int j)
{
    unsigned v[3];
#pragma unroll
    for(int i = 0; i < 3; i++) {
        const uint4_t four = __builtin_bit_cast(uint4_t, q[i]);
        v[i] = j & 1 ? four[j / 2] >> 16 : four[j / 2] & 0xffffu;
    }
    if((v[0] & 0x7f80u) == 0x7f80u)
        return __builtin_bit_cast(float, v[2] << 16 | v[1]);
    return (__builtin_bit_cast(float, v[0] << 16) + __builtin_bit_cast(float, v[1] << 16) + __builtin_bit_cast(float, v[2] << 16)) * SPLIT_DOWN;
}

// acc + low += q * p (times 2^48) over sixteen reduction indices, one product of two parts at a time; rows of the result are q's
constexpr int SPLIT_PRODUCTS = 6;
template <typename V> __device__ __forceinline__ void mfma_split(int j, const Parts &p, const V (&q)[3], float16_t &acc, float16_t &low)
{
    constexpr int qi[] = {0, 1, 0, 1, 2, 0}, pi[] = {0, 0, 1, 1, 0, 2};
    float16_t &to = j ? low : acc;
    to = __builtin_amdgcn_mfma_f32_32x32x16_bf16(part(q[qi[j]]), part(p.v[pi[j]]), to, 0, 0, 0);
}
