// fp32 products on the bf16 matrix cores (gfx950).
//
// An fp32 value is the sum of three bf16 values h + m + l (8 + 8 + 8 significant
// bits, each the rounding of what the ones before it left): exact while l stays
// a normal number, i.e. for |v| >= 2^-110.  A product of two such values is
// taken as the six MFMAs
//   l_a h_b, m_a m_b, h_a l_b, m_a h_b, h_a m_b, h_a h_b
// whose bf16 x bf16 products are exact in fp32; what is left out (m l, l m,
// l l) is below 2^-25 of the product, half an fp32 rounding.  All six add into
// the same fp32 accumulators, the small ones first.  The bf16 pipe runs 16
// times the fp32 one's rate (2.5 PFLOP/s against 157 TFLOP/s dense), so six
// passes still leave 2.7 times the fp32 peak, and one 16-deep MFMA rounds the
// accumulator once where the fp32 instruction rounds it every two products.
#pragma once
#include "kans_common.h"

namespace kans {

typedef float float2_v __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// Two fp32 values as a packed bf16 pair (one v_cvt_pk_bf16_f32).
__device__ __forceinline__ unsigned bf16_pair(float a, float b) {
  const bf16x2 p = __builtin_convertvector((float2_v{a, b}), bf16x2);
  unsigned u;
  __builtin_memcpy(&u, &p, 4);
  return u;
}

// The three bf16 terms of 8 fp32 values, each packed as one MFMA operand.  An
// infinite or NaN value (and a finite one that rounds to infinity in bf16,
// above 3.3895e38) goes into the l term alone: of the six products it then
// enters one, l_a h_b, where h = inf, m = l = 0 would meet zeros and terms of
// the other sign in three more and turn an infinite sum into NaN.
struct Split8 {
  uint4 t[3];
};

__device__ __forceinline__ Split8 split8(const float* v) {
  constexpr float kFiniteMax = 0x1.fep+127f;  // largest bf16
  unsigned d[3][4];
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const float a = v[2 * p], b = v[2 * p + 1];
    const bool fa = __builtin_fabsf(a) <= kFiniteMax, fb = __builtin_fabsf(b) <= kFiniteMax;
    const float ca = fa ? a : 0.0f, cb = fb ? b : 0.0f;
    const unsigned h = bf16_pair(ca, cb);
    const float ra = ca - __uint_as_float(h << 16), rb = cb - __uint_as_float(h & 0xffff0000u);
    const unsigned m = bf16_pair(ra, rb);
    const float sa = ra - __uint_as_float(m << 16), sb = rb - __uint_as_float(m & 0xffff0000u);
    d[0][p] = h;
    d[1][p] = m;
    d[2][p] = bf16_pair(fa ? sa : a, fb ? sb : b);
  }
  Split8 s;
#pragma unroll
  for (int q = 0; q < 3; ++q) s.t[q] = make_uint4(d[q][0], d[q][1], d[q][2], d[q][3]);
  return s;
}

// acc += a * b over the 16-deep contraction of one MFMA, operands in three
// bf16 terms each.
__device__ __forceinline__ floatx16 mma_split(const bf16x8 (&a)[3], const bf16x8 (&b)[3], floatx16 acc) {
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[2], b[0], acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1], b[1], acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[2], acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1], b[0], acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[1], acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[0], acc, 0, 0, 0);
  return acc;
}

// The same with the five small products in an accumulator of their own, 2^-8 of
// the sum: the sum itself is then rounded once per product tile, not six times.
__device__ __forceinline__ void mma_split2(const bf16x8 (&a)[3], const bf16x8 (&b)[3], floatx16& acc, floatx16& small) {
  small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[2], b[0], small, 0, 0, 0);
  small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1], b[1], small, 0, 0, 0);
  small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[2], small, 0, 0, 0);
  small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1], b[0], small, 0, 0, 0);
  small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[1], small, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[0], acc, 0, 0, 0);
}

// The same with a 4:2 sparse left operand of 32 contraction indices (two
// non-zeros in each group of four, their places in the low 16 bits of idx):
// v_smfmac_f32_32x32x32_bf16 takes the time of the 16-deep dense MFMA.
// Lane l of A (row l%32, h = l/32) holds the non-zeros of groups g = 0..3 at
// elements 2g, 2g+1, whose places (0..3 in their group) are bits 4g..4g+1 and
// 4g+2..4g+3 of idx; group g of half h meets elements 8h + 4(g%2) .. +3 of B's
// lane half g/2 (B: column l%32, contraction indices 16(l/32) .. +15).
typedef __bf16 bf16x16 __attribute__((ext_vector_type(16)));
__device__ __forceinline__ floatx16 smfma_split(const bf16x8 (&a)[3], const bf16x16 (&b)[3], int idx, floatx16 acc) {
  acc = __builtin_amdgcn_smfmac_f32_32x32x32_bf16(a[2], b[0], acc, idx, 0, 0);
  acc = __builtin_amdgcn_smfmac_f32_32x32x32_bf16(a[1], b[1], acc, idx, 0, 0);
  acc = __builtin_amdgcn_smfmac_f32_32x32x32_bf16(a[0], b[2], acc, idx, 0, 0);
  acc = __builtin_amdgcn_smfmac_f32_32x32x32_bf16(a[1], b[0], acc, idx, 0, 0);
  acc = __builtin_amdgcn_smfmac_f32_32x32x32_bf16(a[0], b[1], acc, idx, 0, 0);
  acc = __builtin_amdgcn_smfmac_f32_32x32x32_bf16(a[0], b[0], acc, idx, 0, 0);
  return acc;
}

}  // namespace kans
