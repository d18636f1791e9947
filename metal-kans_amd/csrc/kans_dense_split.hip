// Fused forward of fp32 layers on the bf16 matrix cores (kans_split.h: every
// operand in three bf16 terms, six MFMAs per product tile, fp32 accumulation).
//
// Same decomposition as kan_fused_block (kans_dense.hip): a wave owns 32 rows x
// NB*32 output columns, evaluates the basis values of its rows in registers and
// multiplies them by weight fragments from LDS; WAVES waves stack along rows.
// The contraction runs over steps (16-feature block, slot); a step's weights
// are NB tiles of 3 KB (three terms, split once at upload), consecutive steps
// are nob_pad tiles apart also across feature blocks, so the LDS stages hold
// CS consecutive steps whatever the number of slots: two stages, one barrier
// per CS steps, the DMA of the next chunk issued when a chunk begins.
//
// Per wave and step: 6 NB MFMAs (1536 cycles at NB = 8) against 3 NB
// B-fragment reads and about 110 VALU instructions (basis value, split) for
// the next step, a quarter to a half of what the 16-bit kernel spends per MFMA.
// The bound is the MFMA rate that dense mantissas leave: an 8192^3 bf16 product
// reaches 1.12 PFLOP/s on the same card, this kernel 1.24 (six times 206 TFLOP/s
// of fp32 products; the fp32 MFMA's peak is 157).  8192 x 1024 -> 1024, Chebyshev
// K = 4 with the base branch, the four slots left without T_0: 333 us, 582 on the
// fp32 MFMA (118 TFLOP/s).  Layers of about 10 us are up to 2 us slower than on the
// fp32 MFMA (96 x 456 -> 89, K = 6: 10.9 and 9.5): one wave per SIMD waits for the
// split of each step and for 1.5 times the weights.
#include "kans_common.h"
#include "kans_api_internal.h"
#include "kans_split.h"
#include "kans_tile.h"
#include <algorithm>

namespace kans {

// Basis values of 8 inputs in fp32, one basis function after the other.
template <int BASIS> struct SplitBasis;

template <> struct SplitBasis<BASIS_CHEBY> {
  float tw[8], c[8], p[8];  // 2t, T_{k-1}, T_{k-2}
  __device__ __forceinline__ void begin(const float* x, const BasisParams& bp) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float t = __builtin_fminf(__builtin_fmaxf(x[j], -1.0f), 1.0f);
      tw[j] = t + t;
      c[j] = bp.k0 ? 1.0f : t;                              // T_{k0-1}
      p[j] = bp.k0 ? t : __builtin_fmaf(tw[j], t, -1.0f);   // T_{k0-2}
    }
  }
  __device__ __forceinline__ void next(int, const BasisParams&, const float*, float* v) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      v[j] = __builtin_fmaf(tw[j], c[j], -p[j]);
      p[j] = c[j];
      c[j] = v[j];
    }
  }
};

template <> struct SplitBasis<BASIS_RBF> {
  float xv[8];
  __device__ __forceinline__ void begin(const float* x, const BasisParams&) {
#pragma unroll
    for (int j = 0; j < 8; ++j) xv[j] = x[j];
  }
  // tab: the scaled centres in LDS (a scalar load from the argument segment would wait for every LDS read)
  __device__ __forceinline__ void next(int k, const BasisParams& bp, const float* tab, float* v) {
    const float sck = tab[k];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float t = __builtin_fmaf(xv[j], bp.rbf_s, -sck);
      v[j] = __builtin_amdgcn_exp2f(-(t * t));
    }
  }
};

template <> struct SplitBasis<BASIS_BSPLINE> {
  BasisGen<BASIS_BSPLINE, 8> g;
  __device__ __forceinline__ void begin(const float* x, const BasisParams& bp) { g.begin(x, bp); }
  __device__ __forceinline__ void next(int k, const BasisParams& bp, const float*, float* v) { g.one(k, bp, v); }
};

template <int BASIS, int NB, int WAVES, int CS>
__global__ void __launch_bounds__(WAVES * 64, WAVES == 8 ? 1 : 2)
kan_fused_split(const float* __restrict__ X, long ldx, const uint4* __restrict__ Wt, int nob_pad,
                const float* __restrict__ bias, float* __restrict__ Y, long ldy, float* __restrict__ Ypart, int B,
                int D_in, int D_out, int m_tiles, int n_tiles, int nfb_total, int fb_per_split, int has_base,
                BasisParams bp) {
  constexpr int STEP = NB * 192;  // uint4 per step: NB tiles of 3 terms x 64 lanes
  __shared__ uint4 stage0[CS * STEP], stage1[CS * STEP];
  __shared__ float rbf_tab[BASIS == BASIS_RBF ? kMaxK : 1];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int m_tile, n_tile;
  tile_of(xcd_remap(blockIdx.x, m_tiles * n_tiles), m_tiles, n_tiles, m_tile, n_tile);
  const int split = blockIdx.y;
  const int row0 = (m_tile * WAVES + wave) * 32;
  const int ob0 = n_tile * NB;
  const int fb_begin = split * fb_per_split, fb_end = min(nfb_total, fb_begin + fb_per_split);
  if (fb_end <= fb_begin) return;  // uniform per workgroup (empty split)
  const int KP = bp.K + has_base;
  const int nsteps = (fb_end - fb_begin) * KP;

  const uint4* wsrc = Wt + ((long)fb_begin * KP * nob_pad + ob0) * 192 + lane;
  const long wstep = (long)nob_pad * 192;
  auto dma = [&](int c, uint4* stage) {
    const int n = min(CS, nsteps - c * CS) * NB * 3;
    for (int j = wave; j < n; j += WAVES) {
      const int q = j / (NB * 3);
      __builtin_amdgcn_global_load_lds(wsrc + (c * CS + q) * wstep + (j - q * NB * 3) * 64,
                                       (__attribute__((address_space(3))) void*)(stage + j * 64), 16, 0, 0);
    }
  };
  // x[row0 + lane%32][fb*16 + 8*(lane/32) + j], j = 0..7
  uint4 xr[2];
  auto xload = [&](int fb) {
    const int f0 = fb * 16 + 8 * (lane >> 5), row = row0 + (lane & 31);
    const bool ok = row < B && f0 < D_in;
    const uint4* p = reinterpret_cast<const uint4*>(X + (long)row * ldx + f0);
#pragma unroll
    for (int c = 0; c < 2; ++c) xr[c] = ok ? p[c] : make_uint4(0, 0, 0, 0);
  };
  float xf[8];
  SplitBasis<BASIS> gen;
  auto begin_block = [&](int fb) {
    __builtin_memcpy(xf, xr, 32);
    if ((fb + 1) * 16 > D_in) {  // inputs at or beyond D_in read as 0 whatever the padding holds
      const int f0 = fb * 16 + 8 * (lane >> 5);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (f0 + j >= D_in) xf[j] = 0.0f;
    }
    if (fb + 1 < fb_end) xload(fb + 1);
    gen.begin(xf, bp);
  };
  // A operand of slot s
  auto frags = [&](int s, bf16x8 (&a)[3]) {
    float v[8];
    Split8 t;
    if (has_base && s == 0) {
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = silu_f32(xf[j]);
      t = split8(v);
    } else {
      gen.next(s - has_base, bp, rbf_tab, v);
      t = split8_bounded(v);
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) a[q] = *reinterpret_cast<const bf16x8*>(&t.t[q]);
  };

  // kTwo: the small products in registers of their own (mma_split2), which the
  // 256-column tile has not got; it adds up in runs instead (kRun)
  constexpr bool kTwo = NB <= 4;
  floatx16 acc[NB], small[kTwo ? NB : 1];
  auto clear = [&]() {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        acc[nb][r] = 0.0f;
        if (kTwo) small[nb][r] = 0.0f;
      }
  };
  clear();

  if constexpr (BASIS == BASIS_RBF) {
    if (tid < bp.K) rbf_tab[tid] = bp.rbf_sc[tid];
  }
  dma(0, stage0);
  xload(fb_begin);
  __syncthreads();
  int fb = fb_begin, s = 0;
  bf16x8 a[3];
  {
    begin_block(fb);
    frags(0, a);
  }
  auto chunk = [&](int c, const uint4* cur, uint4* nxt) {
    if ((c + 1) * CS < nsteps) dma(c + 1, nxt);
    const int n = min(CS, nsteps - c * CS);
    for (int q = 0; q < n; ++q) {
      // the next step's basis values (past the last step: unused)
      if (++s == KP) {
        s = 0;
        if (++fb < fb_end) begin_block(fb);
      }
      bf16x8 an[3];
      frags(s, an);
      const uint4* st = cur + q * STEP + lane;
      bf16x8 b[2][3];
      auto bread = [&](int nb) {
#pragma unroll
        for (int p = 0; p < 3; ++p) {
          const uint4 u = st[(nb * 3 + p) * 64];
          b[nb & 1][p] = *reinterpret_cast<const bf16x8*>(&u);
        }
      };
      bread(0);
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        if (nb + 1 < NB) bread(nb + 1);
        if constexpr (kTwo) mma_split2(a, b[nb & 1], acc[nb], small[nb]);
        else acc[nb] = mma_split(a, b[nb & 1], acc[nb]);
      }
#pragma unroll
      for (int p = 0; p < 3; ++p) a[p] = an[p];
    }
    __syncthreads();
  };
  // acc register r of lane l holds row 8*(r/4) + 4*(l/32) + r%4, column l%32.
  // first: the sums so far start at the constant term, else at what the output holds
  auto flush = [&](bool first) {
    int rbase = row0 + 4 * (lane >> 5);
    asm volatile("" : "+v"(rbase));  // opaque: the row addresses are not kept through the steps
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const int col = (ob0 + nb) * 32 + (lane & 31);
      if (col < D_out) {
        // loaded and waited for once, before the row tests (see kan_fused_block)
        float bcol = bias != nullptr && Ypart == nullptr ? bias[col] : 0.0f;
        asm volatile("" : "+v"(bcol));
        float* out = Ypart != nullptr ? Ypart + ((long)split * B + rbase) * D_out + col : Y + (long)rbase * ldy + col;
        const long ld = Ypart != nullptr ? D_out : ldy;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int dr = 8 * (r >> 2) + (r & 3);
          if (rbase + dr < B) {
            float* o = out + dr * ld;
            const float sum = kTwo ? acc[nb][r] + small[nb][r] : acc[nb][r];
            __builtin_nontemporal_store(sum + (first ? bcol : *o), o);
          }
        }
      }
    }
  };
  // The 256-column tile adds a long contraction up in runs of 512 steps, each
  // from zero: the rounding error of a run grows with the square root of its
  // length (RBF, D_in = 4096, 2304 steps: 1.57e-6 of the result, 3.08e-6 on the
  // fp32 MFMA in one run).
  constexpr int kRun = 512;
  const int chunks = (nsteps + CS - 1) / CS;
  bool first = true;
  for (int c = 0, run = 0; c < chunks; c += 2) {
    chunk(c, stage0, stage1);
    if (c + 1 < chunks) chunk(c + 1, stage1, stage0);
    if constexpr (!kTwo) {
      run += 2 * CS;
      if (run >= kRun && c + 2 < chunks) {
        flush(first);
        first = false;
        run = 0;
        clear();
      }
    }
  }
  flush(first);
}

// ---------------------------------------------------------------------------
// B-spline layers with K >= 5 on the sparse matrix instructions.
//
// An input has four non-zero basis functions, span .. span+3, one of each
// residue mod 4: the layout of kSparseSteps (kans_common.h) puts exactly two
// candidates of one input in each group of four contraction indices, so four
// v_smfmac steps contract 8 basis functions of a 16-feature block in the time of
// four dense steps, and round the accumulator half as often (the error against
// 64 bits is below the fp32 MFMA kernel's; eight dense steps of three bf16 terms
// were 15 % above it, as they round at the zeros too).
//
// A chunk is CH sparse steps (the first of a feature block also has the base
// slot): two LDS stages, the next chunk's DMA issued when a chunk begins.
// 8192 x 1024 -> 4096, K = 8 with the base branch: 1839 us, fp32 MFMA 4880 us,
// dense steps of three bf16 terms 2746 us.
// ---------------------------------------------------------------------------
template <int NB, int WAVES, int CH>
__global__ void __launch_bounds__(WAVES * 64, WAVES == 8 ? 1 : 2)
kan_fused_split_sparse(const float* __restrict__ X, long ldx, const uint4* __restrict__ Wt, int nob_pad,
                       const float* __restrict__ bias, float* __restrict__ Y, long ldy, float* __restrict__ Ypart,
                       int B, int D_in, int D_out, int m_tiles, int n_tiles, int nfb_total, int fb_per_split,
                       int has_base, BasisParams bp) {
  constexpr int UNIT = NB * 192;  // uint4 of a base slot; a sparse step has two
  __shared__ uint4 stage0[(1 + 2 * CH) * UNIT], stage1[(1 + 2 * CH) * UNIT];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int m_tile, n_tile;
  tile_of(xcd_remap(blockIdx.x, m_tiles * n_tiles), m_tiles, n_tiles, m_tile, n_tile);
  const int split = blockIdx.y;
  const int row0 = (m_tile * WAVES + wave) * 32;
  const int ob0 = n_tile * NB;
  const int fb_begin = split * fb_per_split, fb_end = min(nfb_total, fb_begin + fb_per_split);
  if (fb_end <= fb_begin) return;  // uniform per workgroup (empty split)
  const int steps = kSparseSteps * sparse_blocks(bp.K), nch = steps / CH;
  const int units = has_base + 2 * steps;

  // chunk ch of feature block fb; one DMA instruction moves 64 uint4
  auto dma = [&](int fb, int ch, uint4* stage) {
    const uint4* src = Wt + (long)fb * units * nob_pad * 192 + lane;
    if (ch == 0 && has_base) {
      for (int j = wave; j < NB * 3; j += WAVES)
        __builtin_amdgcn_global_load_lds(src + ((long)ob0 * 3 + j) * 64,
                                         (__attribute__((address_space(3))) void*)(stage + j * 64), 16, 0, 0);
    }
    src += ((long)(has_base + 2 * ch * CH) * nob_pad + 2 * ob0) * 192;
    for (int j = wave; j < CH * NB * 6; j += WAVES) {
      const int q = j / (NB * 6);
      __builtin_amdgcn_global_load_lds(src + (long)q * 2 * nob_pad * 192 + (j - q * NB * 6) * 64,
                                       (__attribute__((address_space(3))) void*)(stage + UNIT + j * 64), 16, 0, 0);
    }
  };
  // x[row0 + lane%32][fb*16 + 8*(lane/32) + j], j = 0..7
  uint4 xr[2];
  auto xload = [&](int fb) {
    const int f0 = fb * 16 + 8 * (lane >> 5), row = row0 + (lane & 31);
    const bool ok = row < B && f0 < D_in;
    const uint4* p = reinterpret_cast<const uint4*>(X + (long)row * ldx + f0);
#pragma unroll
    for (int c = 0; c < 2; ++c) xr[c] = ok ? p[c] : make_uint4(0, 0, 0, 0);
  };
  float xf[8];
  auto begin_block = [&](int fb) {
    __builtin_memcpy(xf, xr, 32);
    if ((fb + 1) * 16 > D_in) {  // inputs at or beyond D_in read as 0 whatever the padding holds
      const int f0 = fb * 16 + 8 * (lane >> 5);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (f0 + j >= D_in) xf[j] = 0.0f;
    }
    if (fb + 1 < fb_end) xload(fb + 1);
  };
  auto frags = [&](const Split8& t, bf16x8 (&a)[3]) {
#pragma unroll
    for (int q = 0; q < 3; ++q) a[q] = *reinterpret_cast<const bf16x8*>(&t.t[q]);
  };
  // A operand of step st: for each of 4 features the basis functions of residues 2P and 2P+1 mod 4 (zero where
  // they lie in another block of 8) and their places in the group.  BasisGen<BASIS_BSPLINE>'s formulas.
  auto sparse_a = [&](int st, bf16x8 (&a)[3], int& idx) {
    const int m = st >> 2, P = (st >> 1) & 1, fh = st & 1;
    float v[8], lo[4], hi[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      lo[g] = xf[g];
      hi[g] = xf[4 + g];
      // opaque: a select of two array elements became an indexed access and xf an array in LDS
      asm volatile("" : "+v"(lo[g]), "+v"(hi[g]));
    }
    idx = 0;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const float x = fh ? hi[g] : lo[g];
      const float pos = (x - bp.grid_min) * bp.inv_h;
      float fl = __builtin_floorf(pos);
      fl = __builtin_fminf(__builtin_fmaxf(fl, 0.0f), (float)(bp.grid_size - 1));
      const float u = __builtin_fminf(__builtin_fmaxf(pos - fl, 0.0f), 1.0f);
      const float om = 1.0f - u, u2 = u * u, u3 = u2 * u;
      const float inv6 = 1.0f / 6.0f;
      const float w0 = om * om * om * inv6;
      const float w1 = (3.0f * u3 - 6.0f * u2 + 4.0f) * inv6;
      const float w2 = (-3.0f * u3 + 3.0f * u2 + 3.0f * u + 1.0f) * inv6;
      const float w3 = u3 * inv6;
      const int span = (int)fl;
      const int t0 = (2 * P - span) & 3, t1 = (t0 + 1) & 3;  // weights of residues 2P, 2P + 1
      const bool odd = t0 & 1, up = t0 & 2;
      const float v0 = up ? (odd ? w3 : w2) : (odd ? w1 : w0);
      const float v1 = up ? (odd ? w0 : w3) : (odd ? w2 : w1);
      const int k0 = span + t0 - 8 * m, k1 = span + t1 - 8 * m;  // functions, from the block's first
      v[2 * g] = (unsigned)k0 < 8u ? v0 : 0.0f;
      v[2 * g + 1] = (unsigned)k1 < 8u ? v1 : 0.0f;
      idx |= (((k0 >> 2) & 1) | (k1 & 4) | 8) << (4 * g);
    }
    frags(split8_bounded(v), a);
  };

  floatx16 acc[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[nb][r] = 0.0f;

  dma(fb_begin, 0, stage0);
  xload(fb_begin);
  __syncthreads();
  auto chunk = [&](int fb, int ch, const uint4* cur, uint4* nxt) {
    if (ch + 1 < nch) dma(fb, ch + 1, nxt);
    else if (fb + 1 < fb_end) dma(fb + 1, 0, nxt);
    if (ch == 0) {
      begin_block(fb);
      if (has_base) {
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = silu_f32(xf[j]);
        bf16x8 a[3];
        frags(split8(v), a);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          bf16x8 b[3];
#pragma unroll
          for (int p = 0; p < 3; ++p) {
            const uint4 u = cur[(nb * 3 + p) * 64 + lane];
            b[p] = *reinterpret_cast<const bf16x8*>(&u);
          }
          acc[nb] = mma_split(a, b, acc[nb]);
        }
      }
    }
#pragma unroll 1
    for (int q = 0; q < CH; ++q) {
      bf16x8 a[3];
      int idx;
      sparse_a(ch * CH + q, a, idx);
      // the weights are read after the basis values: both at once would spill the sums
      __builtin_amdgcn_sched_barrier(0);
      const uint4* st = cur + UNIT + q * 2 * UNIT + lane;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        bf16x16 b[3];
#pragma unroll
        for (int p = 0; p < 3; ++p) {
          uint4 u[2];
          u[0] = st[(nb * 6 + 2 * p) * 64];
          u[1] = st[(nb * 6 + 2 * p + 1) * 64];
          __builtin_memcpy(&b[p], u, 32);
        }
        acc[nb] = smfma_split(a, b, idx, acc[nb]);
      }
    }
    __syncthreads();
  };
  const int total = (fb_end - fb_begin) * nch;
  int fb = fb_begin, ch = 0;
  auto next = [&]() {
    if (++ch == nch) {
      ch = 0;
      ++fb;
    }
  };
  for (int c = 0; c < total; c += 2) {
    chunk(fb, ch, stage0, stage1);
    next();
    if (c + 1 < total) {
      chunk(fb, ch, stage1, stage0);
      next();
    }
  }

  // acc register r of lane l holds row 8*(r/4) + 4*(l/32) + r%4, column l%32
  const int rbase = row0 + 4 * (lane >> 5);
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const int col = (ob0 + nb) * 32 + (lane & 31);
    if (col < D_out) {
      // loaded and waited for once, before the row tests (see kan_fused_block)
      float bcol = bias != nullptr && Ypart == nullptr ? bias[col] : 0.0f;
      asm volatile("" : "+v"(bcol));
      float* out = Ypart != nullptr ? Ypart + ((long)split * B + rbase) * D_out + col : Y + (long)rbase * ldy + col;
      const long ld = Ypart != nullptr ? D_out : ldy;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int dr = 8 * (r >> 2) + (r & 3);
        if (rbase + dr < B) __builtin_nontemporal_store(acc[nb][r] + bcol, out + dr * ld);
      }
    }
  }
}

// Waves per workgroup of tile (wm, nb); its rows are 32 per wave.
int split_waves(int wm, int nb) { return wm == 64 || nb == 8 ? 8 : 4; }

template <int BASIS, int NB, int WAVES, int CS>
static hipError_t launch_t(const DenseLaunch& L, int splits, int fbps, float* part, hipStream_t st) {
  const int m_tiles = (L.B + 32 * WAVES - 1) / (32 * WAVES);
  const int n_tiles = ((L.D_out + 31) / 32 + NB - 1) / NB;
  hipLaunchKernelGGL((kan_fused_split<BASIS, NB, WAVES, CS>), dim3(m_tiles * n_tiles, splits), dim3(WAVES * 64), 0, st,
                     (const float*)L.X, L.ldx, (const uint4*)L.Wt, L.nob_pad, L.bias, (float*)L.Y, L.ldy, part, L.B,
                     L.D_in, L.D_out, m_tiles, n_tiles, L.nfb, fbps, L.has_base, L.bp);
  return hipGetLastError();
}

// Steps per LDS stage: 72 KB stages with one workgroup per CU, 36 KB with two.
template <int BASIS>
static hipError_t launch_basis(const DenseLaunch& L, int splits, int fbps, float* part, hipStream_t st) {
  if (L.wm == 32 && L.nb == 8) return launch_t<BASIS, 8, 8, 3>(L, splits, fbps, part, st);
  if (L.wm == 64 && L.nb == 4) return launch_t<BASIS, 4, 8, 6>(L, splits, fbps, part, st);
  if (L.wm == 32 && L.nb == 4) return launch_t<BASIS, 4, 4, 3>(L, splits, fbps, part, st);
  if (L.wm == 32 && L.nb == 1) return launch_t<BASIS, 1, 4, 12>(L, splits, fbps, part, st);
  return hipErrorInvalidValue;
}

// Whether an fp32 layer's weights and kernel take the sparse layout.
bool split_sparse(int basis, int K) { return basis == BASIS_BSPLINE && K >= 5; }

template <int NB, int WAVES, int CH>
static hipError_t launch_sparse_t(const DenseLaunch& L, int splits, int fbps, float* part, hipStream_t st) {
  const int m_tiles = (L.B + 32 * WAVES - 1) / (32 * WAVES);
  const int n_tiles = ((L.D_out + 31) / 32 + NB - 1) / NB;
  hipLaunchKernelGGL((kan_fused_split_sparse<NB, WAVES, CH>), dim3(m_tiles * n_tiles, splits), dim3(WAVES * 64), 0, st,
                     (const float*)L.X, L.ldx, (const uint4*)L.Wt, L.nob_pad, L.bias, (float*)L.Y, L.ldy, part, L.B,
                     L.D_in, L.D_out, m_tiles, n_tiles, L.nfb, fbps, L.has_base, L.bp);
  return hipGetLastError();
}

// Steps per LDS stage: 72, 60, 36 (two workgroups per CU) and 27 KB.
static hipError_t launch_sparse(const DenseLaunch& L, int splits, int fbps, float* part, hipStream_t st) {
  if (L.wm == 32 && L.nb == 8) return launch_sparse_t<8, 8, 1>(L, splits, fbps, part, st);
  if (L.wm == 64 && L.nb == 4) return launch_sparse_t<4, 8, 2>(L, splits, fbps, part, st);
  if (L.wm == 32 && L.nb == 4) return launch_sparse_t<4, 4, 1>(L, splits, fbps, part, st);
  if (L.wm == 32 && L.nb == 1) return launch_sparse_t<1, 4, 4>(L, splits, fbps, part, st);
  return hipErrorInvalidValue;
}

hipError_t launch_split(const DenseLaunch& L, int splits, int fbps, float* part, hipStream_t st) {
  switch (L.basis) {
    case BASIS_CHEBY: return launch_basis<BASIS_CHEBY>(L, splits, fbps, part, st);
    case BASIS_RBF: return launch_basis<BASIS_RBF>(L, splits, fbps, part, st);
    default:
      return split_sparse(L.basis, L.bp.K) ? launch_sparse(L, splits, fbps, part, st)
                                           : launch_basis<BASIS_BSPLINE>(L, splits, fbps, part, st);
  }
}

}  // namespace kans
