// fp32 products on the bf16 matrix cores (gfx950).
//
// An fp32 value is the sum of three bf16 values h + m + l (8 + 8 + 8 significant
// bits, each the rounding of what the ones before it left), as in published
// work on products in emulated precision (Henry, Tang and Heinecke, "Leveraging
// the bfloat16 Artificial Intelligence Datatype For Higher-Precision
// Computations", 2019).  Exact for |v| >= 2^-110; smaller values keep all bits
// down to 2^-133, the smallest bf16 number (error at most 2^-134 a value).  A product of two such values is
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

// The three bf16 terms of 8 fp32 values, each packed as one MFMA operand.
struct Split8 {
  uint4 t[3];
};

// Finite values of at most the largest bf16 one (0x1.fep127), and basis values
// (|v| <= 1 or NaN: a NaN makes all three terms NaN).
__device__ __forceinline__ Split8 split8_bounded(const float* v) {
  unsigned d[3][4];
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const float a = v[2 * p], b = v[2 * p + 1];
    const unsigned h = bf16_pair(a, b);
    const float ra = a - __uint_as_float(h << 16), rb = b - __uint_as_float(h & 0xffff0000u);
    const unsigned m = bf16_pair(ra, rb);
    d[0][p] = h;
    d[1][p] = m;
    d[2][p] = bf16_pair(ra - __uint_as_float(m << 16), rb - __uint_as_float(m & 0xffff0000u));
  }
  Split8 s;
#pragma unroll
  for (int q = 0; q < 3; ++q) s.t[q] = make_uint4(d[q][0], d[q][1], d[q][2], d[q][3]);
  return s;
}

// Any fp32 values.  Above the largest bf16 value the h term of a finite one is cut
// off there instead of rounding to infinity; m and l still hold what is left.  An
// infinite or NaN value goes into the l term, with h = +-1 and m = 0: of the six
// products l_a h_b and h_a l_b give the infinite result or the NaN, with the right
// sign also where both values are infinite, and the others stay finite (an infinite
// h would meet terms of the other sign and the zeros of m and l, which turns an
// infinite sum into NaN).  A wave takes this path only if one of its values needs
// it (for all of them it would cost 1.3 % of a training step).
__device__ __forceinline__ Split8 split8(const float* v) {
  constexpr float kMaxBf16 = 0x1.fep+127f;
  float sum = 0.0f;  // of the magnitudes: infinite or NaN if one of them is
#pragma unroll
  for (int j = 0; j < 8; j += 2) sum += __builtin_fabsf(v[j]) + __builtin_fabsf(v[j + 1]);
  if (__builtin_expect(__builtin_amdgcn_ballot_w64(!(sum <= kMaxBf16)) == 0, 1)) return split8_bounded(v);
  float c[8], l[8];
  unsigned d[3][4];
#pragma unroll
  for (int j = 0; j < 8; ++j) c[j] = __builtin_fabsf(v[j]) < __builtin_inff() ? v[j] : __builtin_copysignf(1.0f, v[j]);
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const float a = c[2 * p], b = c[2 * p + 1];
    const unsigned h = bf16_pair(__builtin_amdgcn_fmed3f(a, -kMaxBf16, kMaxBf16), __builtin_amdgcn_fmed3f(b, -kMaxBf16, kMaxBf16));
    const float ra = a - __uint_as_float(h << 16), rb = b - __uint_as_float(h & 0xffff0000u);
    const unsigned m = bf16_pair(ra, rb);
    d[0][p] = h;
    d[1][p] = m;
    l[2 * p] = ra - __uint_as_float(m << 16);
    l[2 * p + 1] = rb - __uint_as_float(m & 0xffff0000u);
  }
#pragma unroll
  for (int j = 0; j < 8; ++j)
    if (!(__builtin_fabsf(v[j]) < __builtin_inff())) l[j] = v[j];
#pragma unroll
  for (int p = 0; p < 4; ++p) d[2][p] = bf16_pair(l[2 * p], l[2 * p + 1]);
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
