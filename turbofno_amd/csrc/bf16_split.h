// fp32 products on the bf16 matrix cores without loss of precision. A float is the exact sum of three bf16 values,
//   x = h + m + l,   h = bf16(x), m = bf16(x - h), l = x - h - m      (round to nearest: |m| <= 2^-8 |x|, |l| <= 2^-16 |x|),
// because a bf16 holds 8 of the 24 significant bits. A product is then formed from six of the nine partial products,
//   x w ~ l h' + h l' + m m' + m h' + h m' + h h'
// the three that are left out (m l', l m', l l') are below 2^-23 |x w| together, half the spacing of floats there. Sums
// are fp32, as in v_mfma_f32_16x16x4_f32, but one instruction adds 32 channels instead of 4, so there are fewer roundings.
// Range: the parts of values below 2^-109 (1.5e-33) reach the smallest bf16 number, 2^-133, so an operand is held to 2^-134
// absolutely there (mode GEMM, K = 64: relative error 1.5e-7 at unit scale, 1.6e-7 at 1e-33, 3.8e-6 at 1e-35, 3.8e-5 at 1e-36; 1.5e-7 at 1e37);
// magnitudes within 2^-9 of the largest float round up to infinity.
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

// the three parts of eight consecutive channels of one row or column: operands of v_mfma_f32_16x16x32_bf16
struct SplitOperand {
    uint4_v h, m, l;
};
// Element j of the two A operand rows of one complex weight times alpha, for a contraction over (re, im) pairs of the other
// operand: (re, -im) gives the real part of the product, (im, re) the imaginary part.
__device__ __forceinline__ void split_weight_rows(float2 w, float2 alpha, SplitOperand& real_row, SplitOperand& imag_row, int j)
{
    unsigned h, m, l;
    split_bf16_pair(w.x * alpha.x - w.y * alpha.y, w.x * alpha.y + w.y * alpha.x, h, m, l);
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
