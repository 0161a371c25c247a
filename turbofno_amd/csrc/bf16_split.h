// fp32 products on the bf16 matrix cores. A float is the exact sum of three bf16 values,
//   x = h + m + l,   h = bf16(x), m = bf16(x - h), l = x - h - m      (round to nearest: |m| <= 2^-8 |x|, |l| <= 2^-17 |x|),
// because a bf16 holds 8 of the 24 significant bits. A product is then formed from six of the nine partial products,
//   x w ~ l h' + h l' + m m' + m h' + h m' + h h'
// the three that are left out (m l', l m', l l') are at most 2^-24 |x w| together, the size of one fp32 rounding. Sums
// are fp32, as in v_mfma_f32_16x16x4_f32, but one instruction adds 32 channels instead of 4, so there are fewer roundings: a sum of
// K = 64 channels is off by 1.5e-7 of itself (2.1e-7 with the fp32 instructions), a single product by up to twice as much as there.
// Six v_mfma_f32_16x16x32_bf16 (16 cycles each) do the work of eight v_mfma_f32_16x16x4_f32 (32 cycles each): 2.7 times the
// rate of the fp32 matrix instructions for the same real product.
#pragma once
#include <hip/hip_runtime.h>

namespace tfno {

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float float2_v __attribute__((ext_vector_type(2)));
typedef float float4_v __attribute__((ext_vector_type(4)));
typedef unsigned uint4_v __attribute__((ext_vector_type(4)));

// two floats -> their three bf16 parts, packed two to a register (a in the low half)
__device__ __forceinline__ void split_bf16_pair(float a, float b, unsigned& h, unsigned& m, unsigned& l)
{
    h = __builtin_bit_cast(unsigned, __builtin_convertvector((float2_v){ a, b }, bf16x2_t));
    float ra = a - __builtin_bit_cast(float, h << 16), rb = b - __builtin_bit_cast(float, h & 0xffff0000u);
    m = __builtin_bit_cast(unsigned, __builtin_convertvector((float2_v){ ra, rb }, bf16x2_t));
    ra -= __builtin_bit_cast(float, m << 16);
    rb -= __builtin_bit_cast(float, m & 0xffff0000u);
    l = __builtin_bit_cast(unsigned, __builtin_convertvector((float2_v){ ra, rb }, bf16x2_t));
}

// Which operands the split holds: zero, and magnitudes from 2^-110 (7.7e-34) to 2^-9 below the largest float. Below 2^-110 the third
// part would need bits under the smallest bf16 number, 2^-133; infinities and the top of the range leave a NaN in the remainder x - h.
// A wave whose operands include such values forms its product again, with fp32 instructions, so that the results have fp32 precision
// and fp32 infinities over the whole range of floats:
//   * small magnitudes are found in the operands: below_split_range(), one minimum per two values, and a second look that tells zeros
//     apart, which are exact; or, where zeros are common, lower(), three instructions per two values without a branch;
//   * the others are found in the accumulators: each leaves a NaN or an infinity in every sum it takes part in.
constexpr float kSplitSmallest = 0x1p-110f;
__device__ __forceinline__ float smaller(float low, float a, float b)
{
    return __builtin_elementwise_minimum(__builtin_elementwise_minimum(low, __builtin_fabsf(a)), __builtin_fabsf(b));
}
__device__ __forceinline__ float smaller(float low, float2 a) { return smaller(low, a.x, a.y); }
// smallest 2 |bits| - 1: a zero wraps to the largest number
constexpr unsigned kSplitLow = (17u << 24) - 1;                  // of 2^-110
__device__ __forceinline__ unsigned lower(unsigned low, float2 v)
{
    const unsigned a = 2u * __builtin_bit_cast(unsigned, v.x) - 1u, b = 2u * __builtin_bit_cast(unsigned, v.y) - 1u;
    const unsigned u = a < b ? a : b;
    return low < u ? low : u;
}
// is the condition true in any lane of the wave: uniform
__device__ __forceinline__ bool any_lane(bool condition) { return __builtin_amdgcn_ballot_w64(condition) != 0; }
// is one of the values small, but not zero, in any lane (a NaN among them hides the others, but not itself from the accumulators)
template <int COUNT> __device__ __forceinline__ bool below_split_range(const float2 (&v)[COUNT])
{
    float low = 1.f;
#pragma unroll
    for (int j = 0; j < COUNT; ++j) low = smaller(low, v[j]);
    if (__builtin_expect(!any_lane(low < kSplitSmallest), 1)) return false;
    unsigned bits = ~0u;
#pragma unroll
    for (int j = 0; j < COUNT; ++j) bits = lower(bits, v[j]);
    return any_lane(bits < kSplitLow);
}
// the largest magnitude so far; NaN stays
__device__ __forceinline__ float larger(float high, float4_v c)
{
    high = __builtin_elementwise_maximum(__builtin_elementwise_maximum(high, __builtin_fabsf(c[0])), __builtin_fabsf(c[1]));
    return __builtin_elementwise_maximum(__builtin_elementwise_maximum(high, __builtin_fabsf(c[2])), __builtin_fabsf(c[3]));
}
__device__ __forceinline__ bool not_finite(float a, float b) { return !(__builtin_elementwise_maximum(a, b) < __builtin_inff()); }

// c += w a in fp32, four channels: one complex value of row (w) and column (a) lane % 16, channel lane / 16, per lane
__device__ __forceinline__ void mac_fp32(float2 w, float2 a, float4_v& re, float4_v& im)
{
    re = __builtin_amdgcn_mfma_f32_16x16x4f32(w.x, a.x, re, 0, 0, 0);
    im = __builtin_amdgcn_mfma_f32_16x16x4f32(w.x, a.y, im, 0, 0, 0);
    re = __builtin_amdgcn_mfma_f32_16x16x4f32(-w.y, a.y, re, 0, 0, 0);
    im = __builtin_amdgcn_mfma_f32_16x16x4f32(w.y, a.x, im, 0, 0, 0);
}

// the three parts of eight consecutive channels of one row or column: operands of v_mfma_f32_16x16x32_bf16
struct SplitOperand {
    uint4_v h, m, l;
};
// Element j of the two A operand rows of one complex weight, for a contraction over (re, im) pairs of the other operand:
// (re, -im) gives the real part of the product, (im, re) the imaginary part.
__device__ __forceinline__ void split_weight_rows(float2 w, SplitOperand& real_row, SplitOperand& imag_row, int j)
{
    unsigned h, m, l;
    split_bf16_pair(w.x, w.y, h, m, l);
    real_row.h[j] = h ^ 0x80000000u; real_row.m[j] = m ^ 0x80000000u; real_row.l[j] = l ^ 0x80000000u;
    imag_row.h[j] = __builtin_amdgcn_alignbit(h, h, 16);
    imag_row.m[j] = __builtin_amdgcn_alignbit(m, m, 16);
    imag_row.l[j] = __builtin_amdgcn_alignbit(l, l, 16);
}
__device__ __forceinline__ float4_v mfma_bf16(uint4_v a, uint4_v b, float4_v c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

// c + a b, smallest products first
__device__ __forceinline__ float4_v mac_split(const SplitOperand& a, const SplitOperand& b, float4_v c)
{
    c = mfma_bf16(a.l, b.h, c);
    c = mfma_bf16(a.h, b.l, c);
    c = mfma_bf16(a.m, b.m, c);
    c = mfma_bf16(a.m, b.h, c);
    c = mfma_bf16(a.h, b.m, c);
    return mfma_bf16(a.h, b.h, c);
}
// c0 += a b0, c1 += a b1: two independent chains
__device__ __forceinline__ void mac_split2(const SplitOperand& a, const SplitOperand& b0, const SplitOperand& b1, float4_v& c0, float4_v& c1)
{
    c0 = mfma_bf16(a.l, b0.h, c0); c1 = mfma_bf16(a.l, b1.h, c1);
    c0 = mfma_bf16(a.h, b0.l, c0); c1 = mfma_bf16(a.h, b1.l, c1);
    c0 = mfma_bf16(a.m, b0.m, c0); c1 = mfma_bf16(a.m, b1.m, c1);
    c0 = mfma_bf16(a.m, b0.h, c0); c1 = mfma_bf16(a.m, b1.h, c1);
    c0 = mfma_bf16(a.h, b0.m, c0); c1 = mfma_bf16(a.h, b1.m, c1);
    c0 = mfma_bf16(a.h, b0.h, c0); c1 = mfma_bf16(a.h, b1.h, c1);
}

// c0 += a0 b, c1 += a1 b: two independent chains
__device__ __forceinline__ void mac_split_pair(const SplitOperand& a0, const SplitOperand& a1, const SplitOperand& b, float4_v& c0, float4_v& c1)
{
    c0 = mfma_bf16(a0.h, b.l, c0); c1 = mfma_bf16(a1.h, b.l, c1);
    c0 = mfma_bf16(a0.l, b.h, c0); c1 = mfma_bf16(a1.l, b.h, c1);
    c0 = mfma_bf16(a0.m, b.m, c0); c1 = mfma_bf16(a1.m, b.m, c1);
    c0 = mfma_bf16(a0.h, b.m, c0); c1 = mfma_bf16(a1.h, b.m, c1);
    c0 = mfma_bf16(a0.m, b.h, c0); c1 = mfma_bf16(a1.m, b.h, c1);
    c0 = mfma_bf16(a0.h, b.h, c0); c1 = mfma_bf16(a1.h, b.h, c1);
}

}  // namespace tfno
