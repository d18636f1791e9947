// Fused Chebyshev KAN layer backward for gfx950, without materialising
// the basis tensor Phi.
//
// Reference: metal_kan_cheby_backward_fused (metal_kan_bridge.mm:4532-4632),
// kernels fused_backward_cheby_dW / fused_backward_cheby_dX
// (fused_kan.metal:2053-2163), and the unfused metal_kan_cheby_backward
// (metal_kan_bridge.mm:2715-2850: Phi in a scratch buffer, MPS GEMMs), which
// computes the same quantities.  For y = bias + SiLU(x) W_base^T + Phi(x) W^T
// and an upstream gradient dY:
//
//   dW[o, i*K+k]  = sum_b dY[b,o] T_k(clamp x[b,i])
//   dW_base[o, i] = sum_b dY[b,o] SiLU(x[b,i])
//   dbias[o]      = sum_b dY[b,o]
//   dX[b, i]      = sum_k (dY W)[b, i*K+k] T'_k(x[b,i]) + (dY W_base)[b,i] SiLU'(x[b,i])
//
// with T'_k taken as 0 where the raw input lies outside [-1, 1] (the clamp is
// flat there).  The reference dW kernel keeps at most 16 coefficients in
// registers; here K goes up to kMaxK.
//
// T_0 = 1 and T'_0 = 0 for every input, so the k = 0 coefficients need no
// contraction: dW[o, i*K] = dbias[o] for every i, and they add nothing to dX.
// The NS = K - 1 + has_base "slots" left are SiLU (when has_base) and
// T_1 .. T_{K-1}.
//
// Both gradients are matrix products on the bf16 matrix cores with every fp32
// operand split into three bf16 terms (kans_split.h: six MFMAs per product
// tile, fp32 accumulation, no operand rounded):
//   * k_cheby_bwd_dw: M = outputs, N = (slot, feature), contraction over the
//     batch; A = dY^T, B = the slot values of x, evaluated in the kernel.
//   * k_cheby_bwd_dx: M = batch rows, N = (slot, feature), contraction over
//     D_out; A = dY, B = the slot weights.  The epilogue multiplies the slot
//     sums of one (row, feature) -- all in one lane -- by T'_k / SiLU' and adds
//     them up.
//
// One workgroup = 8 waves = 4 (M) x 2 (32 features).  A wave owns MB x SG tiles
// of 32 x 32 (MB row blocks, SG slots; MB * SG <= 10 tiles, 160 accumulators).
// Per step of 16 contraction indices every operand tile of the workgroup is
// loaded from global memory, split once by one wave and written to one of two
// LDS stages in MFMA fragment order (3 KB per tile, lane-contiguous 16-byte
// accesses); all waves read their fragments from there.  The two waves of a
// SIMD take turns: one splits the next step's operands (VALU) while the other
// multiplies (MFMA), then they swap, with one barrier per step.  That is
// MB * SG * 6 MFMAs (1536 to 1920 cycles) per wave and step against 150 to 250
// VALU instructions.
//
// The bound is the matrix pipe at 6 x 2 * B * D_in * D_out * NS operations: at
// 8192 x 1024 -> 1024, K = 4 with the base branch, dW takes 346 us and dX 335 us
// (1.19 and 1.23 PFLOP/s of bf16 MFMA; an 8192^3 bf16 product reaches 1.12 on the
// same card), where the fp32 VALU kernels this replaces took 3203 and 2753 us.
// Without the waves' turns 364 and 346 us.
// Grids that leave CUs idle split the contraction (choose_splits) into partial
// sums that a second kernel adds in order: 64 workgroups of dW at that shape
// become 256, and the sums cost 27 us.
//
// 16-bit arrays are read as they are and every gradient is rounded once, from
// its fp32 sum: a dX product is one MFMA, a bf16 dW product four (BwdTerms).
// The steps are too short there for the matrix pipe to be the bound; the loads'
// latency and, in dW, the 43 MB of partial sums are.  2000 x 300 -> 500, K = 6,
// bf16: dW 33 us (41 us with the loads converted as they arrive), its sum 13 us,
// dX 27 us; through fp32 copies of the arrays and back the training step took
// 245 us, now 203 us.
#include "kans_common.h"
#include "kans_api_internal.h"
#include "kans_split.h"
#include "kans_tile.h"
#include <algorithm>
#include <type_traits>

namespace kans {
namespace {

constexpr int kBwdThreads = 512;
constexpr int kBwdF = 64;      // features per workgroup
constexpr int kBwdStep = 16;   // contraction indices per step (one MFMA)
constexpr int kBwdMaxSG = 10;  // slots per workgroup

// T: element type of the layer's arrays (dY, X, W and the gradients).
template <typename T>
struct BwdArgs {
  const T *dY, *X, *W, *Wb;
  T *dW, *dWb, *db, *dX;
  float* part;   // split partial sums (null: one split, results written directly)
  float* dbp;    // split partial sums of dbias
  int B, D_in, D_out, K, has_base, NS;
  int m_tiles, f_tiles, groups;  // of this launch, whose first feature tile is f0
  int f0;
  int steps, steps_per_split;
  int vec;       // dX: rows of dY readable with 16-byte loads
};

// Terms of an operand in LDS.  fp32: the three of kans_split.h.  16-bit layers:
//   dX: dY and W are MFMA operands as they are, one product, exact;
//   dW: dY in bf16 is one bf16 term (a second one holds its infinities and
//       NaNs, which must not meet the zeros among the slot values' lower
//       terms); in fp16 it is split like fp32.  The slot values keep three terms.
template <typename T> struct BwdTerms { static constexpr int dw_a = 3, dx = 1; };
template <> struct BwdTerms<float> { static constexpr int dw_a = 3, dx = 3; };
template <> struct BwdTerms<__bf16> { static constexpr int dw_a = 2, dx = 1; };
template <typename T> struct BwdFrag { typedef typename Mfma<T>::frag frag; };
template <> struct BwdFrag<float> { typedef bf16x8 frag; };

__device__ __forceinline__ float silu_deriv_f32(float x) {
  const float s = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-x * kLog2e));
  return s * (1.0f + x * (1.0f - s));
}

// An operand tile (32 x 16) of a stage: N terms of 64 lanes x 16 bytes, from
// its term `at` on.
__device__ __forceinline__ void put_tile(uint4* stage, int at, int lane, const Split8& s) {
#pragma unroll
  for (int q = 0; q < 3; ++q) stage[(at + q) * 64 + lane] = s.t[q];
}
// bf16 values: the finite ones (+-1 in the others' place, as split8's h), and the others
__device__ __forceinline__ void put_tile_bf16(uint4* stage, int at, int lane, const float* v) {
  unsigned d[2][4];
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const float a = v[2 * p], b = v[2 * p + 1];
    const bool fa = __builtin_fabsf(a) < __builtin_inff(), fb = __builtin_fabsf(b) < __builtin_inff();
    d[0][p] = bf16_pair(fa ? a : __builtin_copysignf(1.0f, a), fb ? b : __builtin_copysignf(1.0f, b));
    d[1][p] = bf16_pair(fa ? 0.0f : a, fb ? 0.0f : b);
  }
#pragma unroll
  for (int q = 0; q < 2; ++q) stage[(at + q) * 64 + lane] = make_uint4(d[q][0], d[q][1], d[q][2], d[q][3]);
}

template <int N, typename Frag>
__device__ __forceinline__ void get_tile(const uint4* stage, int at, int lane, Frag (&f)[N]) {
#pragma unroll
  for (int q = 0; q < N; ++q) {
    const uint4 u = stage[(at + q) * 64 + lane];
    __builtin_memcpy(&f[q], &u, 16);
  }
}

// acc += a b for operands of TA and TB terms (see BwdTerms)
template <typename T, int TA, int TB, typename Frag>
__device__ __forceinline__ floatx16 mma_terms(const Frag (&a)[TA], const Frag (&b)[TB], floatx16 acc) {
  if constexpr (TA == 3 && TB == 3) {
    return mma_split(a, b, acc);
  } else if constexpr (TA == 2 && TB == 3) {
    acc = Mfma<__bf16>::mma(a[1], b[0], acc);
    acc = Mfma<__bf16>::mma(a[0], b[2], acc);
    acc = Mfma<__bf16>::mma(a[0], b[1], acc);
    return Mfma<__bf16>::mma(a[0], b[0], acc);
  } else {
    static_assert(TA == 1 && TB == 1, "terms");
    return Mfma<T>::mma(a[0], b[0], acc);
  }
}

// One step of the wave's MB x SG tiles from a stage (4 MB tiles of A, then the
// 2 x SG of B).
template <typename T, int SG, int MB, int TA, int TB, typename Frag>
__device__ __forceinline__ void multiply(const uint4* stage, int wm, int wf, int lane, floatx16 (&acc)[MB][SG]) {
  Frag a[MB][TA], b[2][TB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) get_tile(stage, (wm * MB + mb) * TA, lane, a[mb]);
  const int b0 = 4 * MB * TA + wf * SG * TB;
  get_tile(stage, b0, lane, b[0]);
#pragma unroll
  for (int s = 0; s < SG; ++s) {
    if (s + 1 < SG) get_tile(stage, b0 + (s + 1) * TB, lane, b[(s + 1) & 1]);
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[mb][s] = mma_terms<T>(a[mb], b[s & 1], acc[mb][s]);
  }
}

template <int SG, int MB>
__device__ __forceinline__ void clear(floatx16 (&acc)[MB][SG]) {
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int s = 0; s < SG; ++s)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[mb][s][r] = 0.0f;
}

template <typename T, int SG, int MB>
__global__ void __launch_bounds__(kBwdThreads) k_cheby_bwd_dw(BwdArgs<T> P) {
  constexpr int NA = 4 * MB, TA = BwdTerms<T>::dw_a;
  __shared__ uint4 stage[2][(NA * TA + 2 * SG * 3) * 64];
  __shared__ float dbs[NA * 32];
  const int lane = threadIdx.x & 63, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave & 3, wf = wave >> 2;

  const int tiles = P.m_tiles * P.f_tiles;
  const int lin = xcd_remap(blockIdx.x, tiles * P.groups);
  const int g = lin / tiles;
  int m_tile, f_tile;
  tile_of(lin - g * tiles, P.m_tiles, P.f_tiles, m_tile, f_tile);
  f_tile += P.f0;
  const int o0 = m_tile * (NA * 32), i0 = f_tile * kBwdF, s0 = g * SG;
  const int split = blockIdx.y;
  const int t0 = split * P.steps_per_split;
  const int nk = min(P.steps - t0, P.steps_per_split);

  // A tiles (dY^T): with MB = 2 one per wave, with MB = 1 one for the waves
  // that evaluate fewer slots
  const bool do_a = MB == 2 || wm >= 2;
  const int a_tile = MB == 2 ? wave : wf * 2 + wm - 2;
  // lanes past D_out / D_in repeat the last one: their sums are not stored
  const int ocol = min(o0 + a_tile * 32 + (lane & 31), P.D_out - 1);
  const int icol = min(i0 + wf * 32 + (lane & 31), P.D_in - 1);
  // as loaded: a conversion here would wait for the loads before the products that hide them
  T la[8], lx[8];
  auto load = [&](int t) {
    const int b0 = (t0 + t) * kBwdStep + 8 * half;
    const T* pa = P.dY + (long)b0 * P.D_out + ocol;
    const T* px = P.X + (long)b0 * P.D_in + icol;
    if ((t0 + t + 1) * kBwdStep <= P.B) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if (do_a) la[j] = pa[(long)j * P.D_out];
        lx[j] = px[(long)j * P.D_in];
      }
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const bool ok = b0 + j < P.B;
        if (do_a) la[j] = ok ? pa[(long)j * P.D_out] : from_f32<T>(0.0f);
        lx[j] = ok ? px[(long)j * P.D_in] : from_f32<T>(0.0f);
      }
    }
  };
  float bsum = 0.0f;  // this lane's share of dbias[ocol]
  const bool base0 = P.has_base != 0 && s0 == 0;
  const int k_first = s0 + 1 - P.has_base;  // T index of the group's first slot (g > 0)
  auto produce = [&](uint4* st) {
    float rx[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) rx[j] = to_f32(lx[j]);
    if (do_a) {
      float ra[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) ra[j] = to_f32(la[j]);
      if constexpr (TA == 2) put_tile_bf16(st, a_tile * TA, lane, ra);
      else put_tile(st, a_tile * TA, lane, split8(ra));
      bsum += ((ra[0] + ra[1]) + (ra[2] + ra[3])) + ((ra[4] + ra[5]) + (ra[6] + ra[7]));
    }
    float tw[8], c[8], p[8];  // 2t, T_k, T_{k-1}
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float t = fminf(fmaxf(rx[j], -1.0f), 1.0f);
      tw[j] = t + t;
      c[j] = t;
      p[j] = 1.0f;
    }
    auto advance = [&]() {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float n = __builtin_fmaf(tw[j], c[j], -p[j]);
        p[j] = c[j];
        c[j] = n;
      }
    };
    for (int k = 1; k < k_first; ++k) advance();
#pragma unroll
    for (int s = 0; s < SG; ++s) {
      const bool mine = (s & 3) == wm;
      if (s == 0 && base0) {
        if (mine) {
          float v[8];
#pragma unroll
          for (int j = 0; j < 8; ++j) v[j] = silu_f32(rx[j]);
          put_tile(st, NA * TA + (wf * SG + s) * 3, lane, split8(v));
        }
      } else {
        if (mine) put_tile(st, NA * TA + (wf * SG + s) * 3, lane, split8_bounded(c));
        if (s + 1 < SG) advance();
      }
    }
  };

  floatx16 acc[MB][SG];
  clear<SG, MB>(acc);
  load(0);
  produce(stage[0]);
  if (nk > 1) load(1);
  __syncthreads();
  for (int t = 0; t < nk; ++t) {
    const uint4* cur = stage[t & 1];
    uint4* nxt = stage[(t + 1) & 1];
    const bool more = t + 1 < nk;
    if (wf == 0 && more) {
      produce(nxt);
      if (t + 2 < nk) load(t + 2);
    }
    multiply<T, SG, MB, TA, 3, bf16x8>(cur, wm, wf, lane, acc);
    if (wf != 0 && more) {
      produce(nxt);
      if (t + 2 < nk) load(t + 2);
    }
    __syncthreads();
  }

  bsum += __shfl_xor(bsum, 32);
  if (do_a && half == 0) dbs[a_tile * 32 + lane] = bsum;
  __syncthreads();
  const int tid = threadIdx.x;
  if (f_tile == 0 && g == 0 && tid < NA * 32 && o0 + tid < P.D_out) {
    if (P.part != nullptr) P.dbp[(long)split * P.D_out + o0 + tid] = dbs[tid];
    else if (P.db != nullptr) P.db[o0 + tid] = from_f32<T>(dbs[tid]);
  }
  // acc register r of lane l holds output 8*(r/4) + 4*(l/32) + r%4, feature l%32
  const int i = i0 + wf * 32 + (lane & 31);
  if (i >= P.D_in) return;
  const long Kd = (long)P.D_in * P.K;
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int ol = (wm * MB + mb) * 32 + 8 * (r >> 2) + 4 * half + (r & 3), o = o0 + ol;
      if (o >= P.D_out) continue;
      if (P.part != nullptr) {
        float* out = P.part + (((long)split * P.D_out + o) * P.NS + s0) * P.D_in + i;
#pragma unroll
        for (int s = 0; s < SG; ++s)
          if (s0 + s < P.NS) out[(long)s * P.D_in] = acc[mb][s][r];
      } else {
        T* out = P.dW + (long)o * Kd + (long)i * P.K;
        if (g == 0) out[0] = from_f32<T>(dbs[ol]);
#pragma unroll
        for (int s = 0; s < SG; ++s) {
          if (s == 0 && base0) P.dWb[(long)o * P.D_in + i] = from_f32<T>(acc[mb][s][r]);
          else if (s0 + s < P.NS) out[s0 + s + 1 - P.has_base] = from_f32<T>(acc[mb][s][r]);
        }
      }
    }
}

// Sum of the splits' partial sums, in split order, into dW / dW_base / dbias.
// One thread per (output, slot, feature); slot 0's threads also write the
// k = 0 coefficient, which is dbias.
template <typename T>
__global__ void k_cheby_bwd_dw_reduce(BwdArgs<T> P, int splits) {
  const long n = (long)P.D_out * P.NS * P.D_in;
  for (long idx = (long)blockIdx.x * blockDim.x + threadIdx.x; idx < n; idx += (long)gridDim.x * blockDim.x) {
    const long row = idx / P.D_in;
    const int i = (int)(idx - row * P.D_in), o = (int)(row / P.NS), sl = (int)(row - (long)o * P.NS);
    float s = 0.0f;
    for (int k0 = 0; k0 < splits; k0 += 8) {
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = k0 + u < splits ? P.part[(long)(k0 + u) * n + idx] : 0.0f;
#pragma unroll
      for (int u = 0; u < 8; ++u) s += v[u];
    }
    T* out = P.dW + ((long)o * P.D_in + i) * P.K;
    if (sl == 0) {
      float d = 0.0f;
      for (int k = 0; k < splits; ++k) d += P.dbp[(long)k * P.D_out + o];
      out[0] = from_f32<T>(d);
      if (i == 0 && P.db != nullptr) P.db[o] = from_f32<T>(d);
    }
    if (sl == 0 && P.has_base) P.dWb[(long)o * P.D_in + i] = from_f32<T>(s);
    else out[sl + 1 - P.has_base] = from_f32<T>(s);
  }
}

// kWide: lane offsets in 64 bits, for rows of W or dY that 32 bits do not reach over (wide_rows).
template <typename T, int SG, int MB, bool kWide>
__global__ void __launch_bounds__(kBwdThreads) k_cheby_bwd_dx(BwdArgs<T> P) {
  typedef typename std::conditional<kWide, size_t, unsigned>::type offset;
  constexpr int NA = 4 * MB, NT = NA + 2 * SG, TT = BwdTerms<T>::dx;
  constexpr int R = (NT + 7) / 8;  // operand tiles a wave loads and splits per step
  __shared__ uint4 stage[2][NT * TT * 64];
  const int lane = threadIdx.x & 63, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave & 3, wf = wave >> 2;

  int m_tile, f_tile;
  tile_of(xcd_remap(blockIdx.x, P.m_tiles * P.f_tiles), P.m_tiles, P.f_tiles, m_tile, f_tile);
  f_tile += P.f0;
  const int b0 = m_tile * (NA * 32), i0 = f_tile * kBwdF;
  const int split = blockIdx.y;
  const int t0 = split * P.steps_per_split;
  const int nk = min(P.steps - t0, P.steps_per_split);
  const long Kd = (long)P.D_in * P.K;
  float* const part = P.part != nullptr ? P.part + (long)split * P.B * P.D_in : nullptr;
  const int i = i0 + wf * 32 + (lane & 31);

  for (int g = 0; g < P.groups; ++g) {
    const int s0 = g * SG;
    // operand tile r * 8 + wave: A (dY rows, contiguous outputs) below NA, else
    // slot weights; lanes past B / D_in and slots past NS repeat the last one
    // (src: the wave's first address, lane_off: this lane's bytes from it)
    const T* src[R];
    offset lane_off[R];
    long stride[R];
    T raw[R][8];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int id = r * 8 + wave;
      const long o = (long)t0 * kBwdStep;
      if (id < NA) {
        const int row = min(b0 + id * 32, P.B - 1);
        src[r] = P.dY + (long)row * P.D_out + o;
        lane_off[r] = (offset)sizeof(T) * ((offset)min(lane & 31, P.B - 1 - row) * P.D_out + 8 * half);
        stride[r] = 1;
      } else {
        const int q = min(id, NT - 1) - NA, f = q / SG;
        const int ic = min(i0 + f * 32 + (lane & 31), P.D_in - 1);
        const int sl = min(s0 + q - f * SG, P.NS - 1), k = sl + 1 - P.has_base;
        const bool base = P.has_base != 0 && sl == 0;
        stride[r] = base ? P.D_in : Kd;
        src[r] = (base ? P.Wb : P.W + k) + o * stride[r];
        lane_off[r] = (offset)sizeof(T) * ((offset)(8 * half) * (offset)stride[r] + (offset)ic * (base ? 1 : P.K));
      }
    }
    auto load = [&](int t) {
      const bool full = (t0 + t + 1) * kBwdStep <= P.D_out;
      const int left = P.D_out - (t0 + t) * kBwdStep - 8 * half;  // outputs from this lane's first on
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int id = r * 8 + wave;
        if (id >= NT) continue;
        const T* p = src[r] + (long)t * kBwdStep * stride[r];
        auto at = [&](int j) { return reinterpret_cast<const T*>(reinterpret_cast<const char*>(p + j * stride[r]) + lane_off[r]); };
        if (full && id < NA && P.vec) {
          constexpr int EPL = 16 / (int)sizeof(T);  // elements of a 16-byte load
#pragma unroll
          for (int q = 0; q < 8 / EPL; ++q) {
            const uint4 u = *reinterpret_cast<const uint4*>(at(q * EPL));
            __builtin_memcpy(&raw[r][q * EPL], &u, 16);
          }
        } else if (full) {
#pragma unroll
          for (int j = 0; j < 8; ++j) raw[r][j] = *at(j);
        } else {
#pragma unroll
          for (int j = 0; j < 8; ++j) raw[r][j] = j < left ? *at(j) : from_f32<T>(0.0f);
        }
      }
    };
    auto produce = [&](uint4* st) {
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (r * 8 + wave < NT) {
          if constexpr (TT == 3) {
            put_tile(st, (r * 8 + wave) * TT, lane, split8(raw[r]));
          } else {
            uint4 u;
            __builtin_memcpy(&u, raw[r], 16);
            st[(r * 8 + wave) * 64 + lane] = u;
          }
        }
    };

    floatx16 acc[MB][SG];
    clear<SG, MB>(acc);
    load(0);
    produce(stage[0]);
    if (nk > 1) load(1);
    __syncthreads();
    for (int t = 0; t < nk; ++t) {
      const uint4* cur = stage[t & 1];
      uint4* nxt = stage[(t + 1) & 1];
      const bool more = t + 1 < nk;
      if (wf == 0 && more) {
        produce(nxt);
        if (t + 2 < nk) load(t + 2);
      }
      multiply<T, SG, MB, TT, TT, typename BwdFrag<T>::frag>(cur, wm, wf, lane, acc);
      if (wf != 0 && more) {
        produce(nxt);
        if (t + 2 < nk) load(t + 2);
      }
      __syncthreads();
    }

    // acc register r of lane l holds row 8*(r/4) + 4*(l/32) + r%4, feature l%32
    const int k_first = max(1, s0 + 1 - P.has_base);
    // opaque, so that the 16 * MB row addresses are not kept in registers through the groups' steps
    int row0 = b0 + wm * MB * 32 + 4 * half;
    asm volatile("" : "+v"(row0));
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      float xs[16];  // one memory round trip per row block
#pragma unroll
      for (int r = 0; r < 16; ++r)
        xs[r] = to_f32(P.X[(long)min(row0 + mb * 32 + 8 * (r >> 2) + (r & 3), P.B - 1) * P.D_in + min(i, P.D_in - 1)]);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int b = row0 + mb * 32 + 8 * (r >> 2) + (r & 3);
        const long at = (long)b * P.D_in + i;
        const float x = xs[r];
        // T'_1 = 1, T'_{k+1} = 2 T_k + 2x T'_k - T'_{k-1}
        float t = x, tp = 1.0f, d = 1.0f, dp = 0.0f;
        auto advance = [&]() {
          const float tn = __builtin_fmaf(2.0f * x, t, -tp);
          const float dn = __builtin_fmaf(2.0f * x, d, __builtin_fmaf(2.0f, t, -dp));
          tp = t;
          t = tn;
          dp = d;
          d = dn;
        };
        for (int k = 1; k < k_first; ++k) advance();
        float dx = 0.0f, poly = 0.0f;
#pragma unroll
        for (int s = 0; s < SG; ++s) {
          if (s == 0 && P.has_base && s0 == 0) {
            dx = acc[mb][s][r] * silu_deriv_f32(x);
          } else if (s0 + s < P.NS) {
            poly = __builtin_fmaf(acc[mb][s][r], d, poly);
            advance();
          }
        }
        if (x >= -1.0f && x <= 1.0f) dx += poly;
        if (b < P.B && i < P.D_in) {
          // several slot groups (fp32 only): each adds to the one before
          if (part != nullptr) part[at] = g == 0 ? dx : part[at] + dx;
          else if constexpr (sizeof(T) == 4) P.dX[at] = g == 0 ? dx : P.dX[at] + dx;
          else P.dX[at] = from_f32<T>(dx);
        }
        // one value at a time: all of them side by side would spill the sums
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
}

template <typename T>
__global__ void k_sum_splits(const float* __restrict__ part, T* __restrict__ out, int splits, long n) {
  for (long idx = (long)blockIdx.x * blockDim.x + threadIdx.x; idx < n; idx += (long)gridDim.x * blockDim.x) {
    float s = 0.0f;
    for (int k0 = 0; k0 < splits; k0 += 8) {
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = k0 + u < splits ? part[(long)(k0 + u) * n + idx] : 0.0f;
#pragma unroll
      for (int u = 0; u < 8; ++u) s += v[u];
    }
    out[idx] = from_f32<T>(s);
  }
}

// K = 1 without the base branch: T_0 alone, dW[o, i] = dbias[o] and dX = 0.
// One workgroup per 64 outputs, four row strides, summed through LDS.
__global__ void __launch_bounds__(256) k_cheby_bwd_const(BwdArgs<float> P) {
  __shared__ float sums[4][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int o = blockIdx.x * 64 + lane;
  float s = 0.0f;
  if (o < P.D_out)
    for (int b = w; b < P.B; b += 4) s += P.dY[(long)b * P.D_out + o];
  sums[w][lane] = s;
  __syncthreads();
  const int o_end = min(P.D_out, (int)(blockIdx.x + 1) * 64);
  for (int q = blockIdx.x * 64 + w; q < o_end; q += 4) {
    const int l = q - blockIdx.x * 64;
    const float d = (sums[0][l] + sums[1][l]) + (sums[2][l] + sums[3][l]);
    if (lane == 0 && P.db != nullptr) P.db[q] = d;
    for (int i = lane; i < P.D_in; i += 64) P.dW[(long)q * P.D_in + i] = d;
  }
}

__global__ void k_fill_zero(float* __restrict__ p, long n) {
  for (long idx = (long)blockIdx.x * blockDim.x + threadIdx.x; idx < n; idx += (long)gridDim.x * blockDim.x) p[idx] = 0.0f;
}

int reduce_blocks(long n) { return (int)std::min<long>((n + 255) / 256, 8192); }

// Contraction splits of a grid of `tiles` workgroups (one per CU at a time, 256
// CUs): the fewest that leave the CUs busy -- a further split has to fill the
// last round of workgroups at least 10 % better -- with at least two steps
// each, and no more than the workspace holds.
int choose_splits(long tiles, int steps, long max_by_ws) {
  auto fill = [&](long s) { return (double)(tiles * s) / (double)((tiles * s + 255) / 256 * 256); };
  const long smax = std::min<long>({64, steps / 2, max_by_ws});
  long best = 1;
  for (long s = 2; s <= smax; ++s)
    if (fill(s) > 1.1 * fill(best)) best = s;
  return (int)best;
}

// Whether the dX kernel's 32-bit lane offsets fall short: 36 bytes a reduction index of W, 124 bytes an output of dY.
bool wide_rows(int D_in, int D_out, int K) { return (long)D_in * K > (1L << 26) || D_out > (1 << 25); }

struct BwdPlan {
  int SG, MB, groups, NS;
  bool wide;
  int splits_w, splits_x;
  size_t ws_floats;
  bool fits;  // a grid holds the workgroups of one feature tile
};

// Workgroups of one launch: a grid holds fewer than 2^32 threads along x.
constexpr long kBwdMaxGrid = 1L << 22;

// Workspace cap of the split partial sums (floats).
constexpr size_t kBwdWsFloats = size_t(64) << 20;

BwdPlan plan_backward(int B, int D_in, int D_out, int K, int has_base, bool may_split) {
  BwdPlan p{};
  p.NS = K - 1 + has_base;
  // (wide rows: one instantiation of the dX kernel, slot by slot)
  p.wide = wide_rows(D_in, D_out, K);
  p.groups = p.wide ? std::max(1, p.NS) : std::max(1, (p.NS + kBwdMaxSG - 1) / kBwdMaxSG);
  p.SG = std::max(1, (p.NS + p.groups - 1) / p.groups);
  p.MB = p.SG <= 5 ? 2 : 1;
  const int M = 4 * p.MB * 32;
  const long f_tiles = (D_in + kBwdF - 1) / kBwdF;
  const long per_w = (long)D_out * ((long)p.NS * D_in + 1), per_x = (long)B * D_in;
  p.fits = ((long)D_out + M - 1) / M * p.groups <= kBwdMaxGrid && ((long)B + M - 1) / M <= kBwdMaxGrid;
  const long cap = may_split ? (long)kBwdWsFloats : 0;
  p.splits_w = choose_splits(((D_out + M - 1) / M) * f_tiles * p.groups, (B + kBwdStep - 1) / kBwdStep, cap / per_w);
  p.splits_x = choose_splits(((B + M - 1) / M) * f_tiles, (D_out + kBwdStep - 1) / kBwdStep, cap / per_x);
  p.ws_floats = std::max(p.splits_w > 1 ? (size_t)(per_w * p.splits_w) : 0,
                         p.splits_x > 1 ? (size_t)(per_x * p.splits_x) : 0);
  return p;
}

template <typename T, int SG, int MB, bool kWide = false>
hipError_t launch_bwd(BwdArgs<T> A, const BwdPlan& p, float* ws, hipStream_t st) {
  constexpr int M = 4 * MB * 32;
  A.groups = p.groups;
  const int f_tiles = (A.D_in + kBwdF - 1) / kBwdF;
  // launch(first feature tile, feature tiles) in parts of at most kBwdMaxGrid workgroups, `per` to a feature tile
  auto parts = [&](long per, auto launch) {
    const int n = (int)std::min<long>(f_tiles, std::max(1L, kBwdMaxGrid / per));
    hipError_t e = hipSuccess;
    for (int f = 0; f < f_tiles && e == hipSuccess; f += n) {
      launch(f, std::min(n, f_tiles - f));
      e = hipGetLastError();
    }
    return e;
  };
  // dW: outputs x (slot, feature), contraction over the batch
  BwdArgs<T> W = A;
  W.m_tiles = (A.D_out + M - 1) / M;
  W.steps = (A.B + kBwdStep - 1) / kBwdStep;
  W.steps_per_split = (W.steps + p.splits_w - 1) / p.splits_w;
  const int splits_w = (W.steps + W.steps_per_split - 1) / W.steps_per_split;
  W.part = splits_w > 1 ? ws : nullptr;
  W.dbp = splits_w > 1 ? ws + (size_t)splits_w * A.D_out * A.NS * A.D_in : nullptr;
  hipError_t e = parts((long)W.m_tiles * A.groups, [&](int f0, int n) {
    W.f0 = f0;
    W.f_tiles = n;
    hipLaunchKernelGGL((k_cheby_bwd_dw<T, SG, MB>), dim3(W.m_tiles * n * A.groups, splits_w), dim3(kBwdThreads), 0, st, W);
  });
  if (e != hipSuccess) return e;
  if (splits_w > 1) {
    hipLaunchKernelGGL((k_cheby_bwd_dw_reduce<T>), dim3(reduce_blocks((long)A.D_out * A.NS * A.D_in)), dim3(256), 0, st, W,
                       splits_w);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  // dX: batch rows x (slot, feature), contraction over the outputs
  BwdArgs<T> X = A;
  X.m_tiles = (A.B + M - 1) / M;
  X.steps = (A.D_out + kBwdStep - 1) / kBwdStep;
  X.steps_per_split = (X.steps + p.splits_x - 1) / p.splits_x;
  const int splits_x = (X.steps + X.steps_per_split - 1) / X.steps_per_split;
  X.part = splits_x > 1 ? ws : nullptr;
  X.vec = A.D_out % (16 / (int)sizeof(T)) == 0 && ((uintptr_t)A.dY & 15) == 0;
  e = parts(X.m_tiles, [&](int f0, int n) {
    X.f0 = f0;
    X.f_tiles = n;
    hipLaunchKernelGGL((k_cheby_bwd_dx<T, SG, MB, kWide>), dim3(X.m_tiles * n, splits_x), dim3(kBwdThreads), 0, st, X);
  });
  if (e != hipSuccess) return e;
  if (splits_x > 1) {
    const long n = (long)A.B * A.D_in;
    hipLaunchKernelGGL((k_sum_splits<T>), dim3(reduce_blocks(n)), dim3(256), 0, st, ws, A.dX, splits_x, n);
    e = hipGetLastError();
  }
  return e;
}


template <typename T>
hipError_t launch_slots(const BwdArgs<T>& A, const BwdPlan& p, float* ws, hipStream_t st) {
  if constexpr (sizeof(T) == 4) {
    if (p.wide) return launch_bwd<T, 1, 2, true>(A, p, ws, st);
  }
  switch (p.SG) {
    case 1: return launch_bwd<T, 1, 2>(A, p, ws, st);
    case 2: return launch_bwd<T, 2, 2>(A, p, ws, st);
    case 3: return launch_bwd<T, 3, 2>(A, p, ws, st);
    case 4: return launch_bwd<T, 4, 2>(A, p, ws, st);
    case 5: return launch_bwd<T, 5, 2>(A, p, ws, st);
    case 6: return launch_bwd<T, 6, 1>(A, p, ws, st);
    case 7: return launch_bwd<T, 7, 1>(A, p, ws, st);
    case 8: return launch_bwd<T, 8, 1>(A, p, ws, st);
    case 9: return launch_bwd<T, 9, 1>(A, p, ws, st);
    default: return launch_bwd<T, 10, 1>(A, p, ws, st);
  }
}

}  // namespace

// ws: p.ws_floats floats when the plan splits, else unused.
template <typename T>
static hipError_t launch_cheby_backward(const void* dY, const void* X, const void* W, const void* Wb, void* dW,
                                        void* dWb, void* db, void* dX, int B, int D_in, int D_out, int K,
                                        int has_base, const BwdPlan& p, float* ws, hipStream_t st) {
  BwdArgs<T> A{};
  A.dY = (const T*)dY; A.X = (const T*)X; A.W = (const T*)W; A.Wb = (const T*)Wb;
  A.dW = (T*)dW; A.dWb = (T*)dWb; A.db = (T*)db; A.dX = (T*)dX;
  A.B = B; A.D_in = D_in; A.D_out = D_out; A.K = K; A.has_base = has_base; A.NS = p.NS;
  if constexpr (sizeof(T) == 4) {
    if (p.NS == 0) {
      hipLaunchKernelGGL(k_cheby_bwd_const, dim3((D_out + 63) / 64), dim3(256), 0, st, A);
      hipError_t e = hipGetLastError();
      if (e != hipSuccess) return e;
      const long n = (long)B * D_in;
      hipLaunchKernelGGL(k_fill_zero, dim3(reduce_blocks(n)), dim3(256), 0, st, (float*)dX, n);
      return hipGetLastError();
    }
  }
  return launch_slots<T>(A, p, ws, st);
}

}  // namespace kans

using namespace kans;

namespace {

// The plan of one backward and the stream's workspace for its partial sums; without one the plan without splits.
int acquire_ws(int B, int D_in, int D_out, int K, int has_base, bool may_split, hipStream_t st, BwdPlan* plan,
                float** ws) {
  *ws = nullptr;
  *plan = plan_backward(B, D_in, D_out, K, has_base, may_split);
  if (!plan->fits)
    return kans_fail(KANS_ERR_UNSUPPORTED, "B=%d or D_out=%d at K=%d: more tiles than a grid holds", B, D_out, K);
  if (plan->ws_floats == 0) return 0;
  *ws = kans_stream_workspace(st, plan->ws_floats * sizeof(float));
  if (!*ws) *plan = plan_backward(B, D_in, D_out, K, has_base, false);
  return 0;
}

int check_bwd(const void* dY, const void* X, const void* W, const void* Wb, const void* dW, const void* dWb,
              const void* dX, int B, int D_in, int D_out, int K, int has_base, int has_bias) {
  if (!dY || !X || !W || !dW || !dX) return kans_fail(KANS_ERR_ARG, "null dY, X, W, dW or dX");
  if (B <= 0 || D_in <= 0 || D_out <= 0 || K <= 0 || K > kMaxK)
    return kans_fail(KANS_ERR_ARG, "bad dims B=%d D_in=%d D_out=%d K=%d (1 <= K <= %d)", B, D_in, D_out, K, kMaxK);
  if ((has_base != 0 && has_base != 1) || (has_bias != 0 && has_bias != 1))
    return kans_fail(KANS_ERR_ARG, "has_base / has_bias must be 0 or 1");
  if (has_base && (!Wb || !dWb)) return kans_fail(KANS_ERR_ARG, "has_base=1 but W_base or dW_base is null");
  return 0;
}

// Host-pointer backward: stage through device buffers, run, copy the gradients back.
int backward_host(const float* dY, const float* X, const float* W, const float* Wb, float* dW, float* dWb,
                  float* db, float* dX, int B, int D_in, int D_out, int K, int has_base, int has_bias) {
  int rc = check_bwd(dY, X, W, Wb, dW, dWb, dX, B, D_in, D_out, K, has_base, has_bias);
  if (rc) return rc;
  if (has_bias && !db) return kans_fail(KANS_ERR_ARG, "has_bias=1 but dbias is null");
  std::lock_guard<std::mutex> lk(kans_mutex());
  if ((rc = kans_ensure_init())) return rc;
  static DevBuf buf;
  const size_t nY = (size_t)B * D_out, nX = (size_t)B * D_in, nW = (size_t)D_out * D_in * K,
               nWb = has_base ? (size_t)D_out * D_in : 0, nb = has_bias ? (size_t)D_out : 0;
  const size_t total = nY + 2 * nX + 2 * nW + 2 * nWb + nb;
  if ((rc = buf.reserve(total * sizeof(float)))) return rc;
  float* p = (float*)buf.p;
  float *d_dY = p, *d_X = d_dY + nY, *d_W = d_X + nX, *d_Wb = d_W + nW, *d_dW = d_Wb + nWb,
        *d_dWb = d_dW + nW, *d_db = d_dWb + nWb, *d_dX = d_db + nb;
  hipStream_t st = kans_default_stream();
  HIP_TRY(hipMemcpyAsync(d_dY, dY, nY * 4, hipMemcpyHostToDevice, st));
  HIP_TRY(hipMemcpyAsync(d_X, X, nX * 4, hipMemcpyHostToDevice, st));
  HIP_TRY(hipMemcpyAsync(d_W, W, nW * 4, hipMemcpyHostToDevice, st));
  if (has_base) HIP_TRY(hipMemcpyAsync(d_Wb, Wb, nWb * 4, hipMemcpyHostToDevice, st));
  BwdPlan plan;
  float* ws;
  if ((rc = acquire_ws(B, D_in, D_out, K, has_base, true, st, &plan, &ws))) return rc;
  HIP_TRY(launch_cheby_backward<float>(d_dY, d_X, d_W, has_base ? d_Wb : nullptr, d_dW, has_base ? d_dWb : nullptr,
                                has_bias ? d_db : nullptr, d_dX, B, D_in, D_out, K, has_base, plan, ws, st));
  HIP_TRY(hipMemcpyAsync(dW, d_dW, nW * 4, hipMemcpyDeviceToHost, st));
  if (has_base) HIP_TRY(hipMemcpyAsync(dWb, d_dWb, nWb * 4, hipMemcpyDeviceToHost, st));
  if (has_bias) HIP_TRY(hipMemcpyAsync(db, d_db, nb * 4, hipMemcpyDeviceToHost, st));
  HIP_TRY(hipMemcpyAsync(dX, d_dX, nX * 4, hipMemcpyDeviceToHost, st));
  HIP_TRY(hipStreamSynchronize(st));
  return 0;
}

}  // namespace

extern "C" {

int kans_cheby_backward_ex(int dtype, const void* dY, const void* X, const void* W, const void* W_base, void* dW,
                           void* dW_base, void* dbias, void* dX, int B, int D_in, int D_out, int K, int has_base,
                           int has_bias, void* stream) {
  int rc = check_bwd(dY, X, W, W_base, dW, dW_base, dX, B, D_in, D_out, K, has_base, has_bias);
  if (rc) return rc;
  if (dtype != DT_F32 && dtype != DT_F16 && dtype != DT_BF16) return kans_fail(KANS_ERR_ARG, "unknown dtype %d", dtype);
  // partial gradients of several slot groups are added up in the output, which has to hold fp32
  if (dtype != DT_F32 && (K - 1 + has_base < 1 || K - 1 + has_base > kBwdMaxSG || wide_rows(D_in, D_out, K)))
    return kans_fail(KANS_ERR_UNSUPPORTED,
                     "16-bit backward takes 1 to %d slots, D_in * K <= 2^26 and D_out <= 2^25 (K - 1 + has_base = %d, "
                     "D_in = %d, D_out = %d)", kBwdMaxSG, K - 1 + has_base, D_in, D_out);
  std::lock_guard<std::mutex> lk(kans_mutex());
  if ((rc = kans_ensure_init())) return rc;
  hipStream_t st = kans_caller_stream(stream);
  // a call recorded into a graph outlives this one: it gets no share of the stream's workspace
  bool capturing = false;
  HIP_TRY(kans_capturing(st, &capturing));
  BwdPlan plan;
  float* ws;
  if ((rc = acquire_ws(B, D_in, D_out, K, has_base, !capturing, st, &plan, &ws))) return rc;
  auto* go = dtype == DT_F16 ? launch_cheby_backward<_Float16>
             : dtype == DT_BF16 ? launch_cheby_backward<__bf16>
                                : launch_cheby_backward<float>;
  HIP_TRY(go(dY, X, W, has_base ? W_base : nullptr, dW, has_base ? dW_base : nullptr, has_bias ? dbias : nullptr, dX, B,
             D_in, D_out, K, has_base, plan, ws, st));
  return 0;
}

int kans_cheby_backward(const float* dY, const float* X, const float* W, const float* W_base, float* dW,
                        float* dW_base, float* dbias, float* dX, int B, int D_in, int D_out, int K, int has_base,
                        int has_bias, void* stream) {
  return kans_cheby_backward_ex(DT_F32, dY, X, W, W_base, dW, dW_base, dbias, dX, B, D_in, D_out, K, has_base, has_bias,
                                stream);
}

int metal_kan_cheby_backward_fused(const float* dY, const float* X, const float* W_cheby, const float* W_base,
                                   float* dW_cheby, float* dW_base, float* dbias, float* dX, int B, int D_in,
                                   int D_out, int degree, int has_base, int has_bias) {
  return backward_host(dY, X, W_cheby, W_base, dW_cheby, dW_base, dbias, dX, B, D_in, D_out, degree, has_base,
                       has_bias);
}

int metal_kan_cheby_backward(const float* dY, const float* X, const float* W_cheby, const float* W_base,
                             float* dW_cheby, float* dW_base, float* dbias, float* dX, int B, int D_in, int D_out,
                             int degree, int has_base, int has_bias) {
  return backward_host(dY, X, W_cheby, W_base, dW_cheby, dW_base, dbias, dX, B, D_in, D_out, degree, has_base,
                       has_bias);
}

}  // extern "C"
