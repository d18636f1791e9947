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

// What is left of v after its bf16 rounding hf.  An infinite or NaN hf leaves
// nothing: the product then is what h alone gives (inf - inf would turn an
// infinity into NaN).
__device__ __forceinline__ float bf16_rest(float v, float hf) {
  const float r = v - hf;
  return __builtin_fabsf(hf) < __builtin_inff() ? r : 0.0f;
}

// The three bf16 terms of 8 fp32 values, each packed as one MFMA operand.
struct Split8 {
  uint4 t[3];
};

__device__ __forceinline__ Split8 split8(const float* v) {
  unsigned d[3][4];
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const float a = v[2 * p], b = v[2 * p + 1];
    const unsigned h = bf16_pair(a, b);
    const float ra = bf16_rest(a, __uint_as_float(h << 16));
    const float rb = bf16_rest(b, __uint_as_float(h & 0xffff0000u));
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

}  // namespace kans
