// Logistic potential + adjoint for fp32 and fp8 designs on the matrix cores,
// C chains.
//
// Same mathematics and work split as the bf16 kernel (logistic_mfma.hip): per
// 32-row tile of X and wave of 32 chains
//   GEMM1  L = X Z^T,  epilogue R = sigmoid(L) - y,  GEMM2  G^T += R^T X,
// with the accumulator of GEMM1 (lane (c, h), register v: row
// 8(v/4) + 4h + v%4 of chain c) being GEMM2's A operand.
//
// GEMM1 runs on the fp32 MFMA, whose accumulation is the chain of fp32 fused
// multiply-adds over d = 0, 1, ... (v_mfma_f32_32x32x2_f32 against fmaf on
// 200,000 random triples: every one equal): logits are those of the VALU tile
// kernel bit for bit.  (Energies are not: the fp32 forms take a row's loss from
// logit_terms and add a lane's 16 rows of a tile in fp32 before the compensated
// fp64 sum, fp8 takes log1p_unit and adds every row in fp64.)  A design in fp8
// codes enters as its code values (exact), its power-of-two column scales go to z.
//
// GEMM2 runs on the fp16 MFMA, which takes 1/16 of the time.  X' (the scaled
// column) is two fp16 terms, hi + lo, and R' = 2^14 r three: a + (b + c) / 2^10.
// hi and a lie on grids (X': 2^-11 of the power of two above the column's rms, R':
// 2^-10 of |r| = 1), because the eight products that the fp16 MFMA adds at once
// are cut (toward zero) 24 bits below the largest, which would add up where r x is
// skewed: products a hi are multiples of one step, and nothing of them is cut.
// b + c hold r - a to 22 bits of itself, for residuals down to 2^-26: with one term
// below the grid a residual under 2^-11 (rare events) had 11 bits, and since
// thousands of rows with the same covariates share it, their errors added up (error
// of 1e-3 below).  The products with b and c are summed from zero over a tile and
// added to the running sum once, so that they do not meet a large sum one by
// one.  Five MFMAs a k-step (fp8 codes are exact in one term: three).  Gradient
// error against float64 over the root of the sum of (r x)^2, rms over 256 chains
// near the generating coefficients, both products on the fp32 MFMA / this / one
// term below R's grid:
//   581,012 x 55, covtype-like             2.3e-6 / 2.3e-6 / 2.3e-6
//   500,000 x 250, normal                  1.4e-6 / 0.9e-6 / 1.3e-6
//   1,000,000 rows in 8 categories, events at 1e-2   5.7e-5 / 6.9e-6 / 1.6e-4
//                                              1e-3   5.2e-5 / 5.3e-6 / 3.4e-4
//                                              1e-4   3.9e-5 / 2.0e-6 / 7.4e-4
//   500,000 x 12 binary, intercept -7      2.3e-5 / 1.5e-6 / 1.8e-4
//   the same, columns standardised         7.1e-5 / 6.8e-6 / 1.5e-4
// (GEMM1 does not take the split: an error of z shifts every row's logit
// alike, and near the mode the gradient answers to it sqrt(N) times over.)
//
// Ranges.  fp16 spans 2^-24 .. 2^16, so the factors are scaled by powers of
// two (exact): column d of X such that max |X'_d| lies in [2^14, 2^15), R by
// 2^14.  A term of 2^-39 of its column's largest is then still represented.
// The split takes a design whose columns are finite with max |X_d| <= 2^12
// rms(X_d), so that this is below fp32's own rounding of a typical element, and
// labels in [0, 1] (|r| <= 1; fp16 ends at |R'| = 2^16).
// Its number of rows is bounded too.  On more than kSplitRows rows per partial
// sum the fp32 accumulators' own rounding is what a result's error consists of,
// and the two forms round differently: the split's error is half the fp32 form's
// (N = 2,000,000, 1024 chains: 4e-6 and 1.4e-5 of the gradient's norm, 12.9 and 16.6
// ms), but their results differ by the larger, so such designs keep the form that
// they have had.  Below kSplitMin rows a launch is mostly latency and the split
// gains little or nothing (256 chains: 16,000 x 55 34.8 against 31.6 us in fp32,
// 16,000 x 200 62 against 69, 65,536 x 100 80 against 96).  Other designs take the
// fp32 MFMA in GEMM2 too.
//
// Bound: MFMA issue (D = 256: GEMM1 8192 cycles per tile and wave, GEMM2 2560
// split, 8192 in fp32) plus the epilogue's VALU work, which the fp32 MFMA hardly
// overlaps (standing between the MFMAs or in groups of its own it takes the same
// time); two blocks share a CU where the registers allow, so that one's GEMM2
// runs beside the other's epilogue.  Main kernel, both products in fp32 and
// split: 581,012 x 55, 256 chains 412 and 319 us (281 with one term below R's grid);
// 500,000 x 250, 256 chains 1.06 and 0.85 ms (0.76); fp8 500,000 x 250, 250 chains
// 13.3 ms on the VALU tile kernel and 0.94 (0.81).  2,000,000 x 256, 1024 chains
// (fp32 form) 17.0 ms with the epilogue between the products, 16.5 as here.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <string>

#include "nax_device.h"
#include "nax_internal.h"

namespace nax {

typedef __attribute__((__vector_size__(8 * sizeof(_Float16)))) _Float16 f16x8;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

constexpr float kRScale = 16384.0f;  // 2^14: |R'| <= 2^14
constexpr float kRFine = 1024.0f;    // of the terms below R's grid
constexpr int64_t kSplitRows = 32768, kSplitMin = 65536;

// hi (on a grid of step q, a power of two, where fp16 is finer) + lo of a
// value already scaled into fp16's range.
__device__ __forceinline__ void split16(float v, float q, _Float16& hi, _Float16& lo) {
  const float m = 12582912.0f * q;  // 1.5 2^23 q: rounds v to a multiple of q
  hi = (_Float16)((v + m) - m);
  lo = (_Float16)(v - (float)hi);
}
constexpr float kRGrid = kRScale / 1024.0f;

// ---- set-up ------------------------------------------------------------------------

constexpr int kStatBlocks = 256;

// Per column and block: the largest |x| as bits (infinities and NaN above every
// finite value) and the sum of squares; blocks take contiguous row ranges.
__global__ void __launch_bounds__(256)
split_col_stats(const float* __restrict__ X, int64_t N, int D, unsigned* __restrict__ pmax,
                double* __restrict__ psq) {
  __shared__ unsigned smax[256];
  __shared__ double ssq[256];
  int dp2 = 1;
  while (dp2 < D) dp2 <<= 1;  // D <= 256
  const int nq = 256 / dp2, q = threadIdx.x / dp2, d = threadIdx.x % dp2;
  const int64_t n0 = N * blockIdx.x / gridDim.x, n1 = N * (blockIdx.x + 1) / gridDim.x;
  unsigned m = 0;
  double s = 0.0;
  if (d < D)
#pragma unroll 8
    for (int64_t n = n0 + q; n < n1; n += nq) {
      const float v = X[n * D + d];
      m = max(m, __float_as_uint(v) & 0x7FFFFFFFu);
      s += (double)v * v;
    }
  smax[threadIdx.x] = m;
  ssq[threadIdx.x] = s;
  __syncthreads();
  if (q == 0 && d < D) {
    for (int k = 1; k < nq; ++k) {
      m = max(m, smax[k * dp2 + d]);
      s += ssq[k * dp2 + d];
    }
    pmax[(size_t)blockIdx.x * D + d] = m;
    psq[(size_t)blockIdx.x * D + d] = s;
  }
}

// cscale[d] = 2^e with max |X_d| 2^-e in [2^14, 2^15) (1 for a zero column) and
// the scaled column's grid cgrid[d]; *bad counts the columns outside the range
// rule.
__global__ void __launch_bounds__(256)
split_col_scale(const unsigned* __restrict__ pmax, const double* __restrict__ psq, int nb,
                int64_t N, int D, float* __restrict__ cscale,
                float* __restrict__ cgrid, int* __restrict__ bad) {
  const int d = threadIdx.x;
  if (d >= D) return;
  unsigned m = 0;
  double s = 0.0;
#pragma unroll 8
  for (int b = 0; b < nb; ++b) {
    m = max(m, pmax[(size_t)b * D + d]);
    s += psq[(size_t)b * D + d];
  }
  const float mx = __uint_as_float(m);
  float sc = 1.0f;
  bool ok = m < 0x7F800000u;
  if (ok && m > 0) {
    int e;
    frexpf(mx, &e);  // mx = f 2^e, f in [0.5, 1)
    sc = ldexpf(1.0f, e - 15);
    ok = (double)mx * mx <= 16777216.0 * (s / (double)N) && e - 15 >= -125;
  }
  cscale[d] = sc;
  int e = 0;
  if (ok) frexp(sqrt(s / (double)N) / sc, &e);  // rms of the scaled column in [2^(e-1), 2^e)
  cgrid[d] = ldexpf(1.0f, e - 11);
  if (!ok) atomicAdd(bad, 1);
}

// Adds the labels outside [0, 1] to *bad: a residual of 4 or more is past fp16
// after R's scale.
__global__ void __launch_bounds__(256)
split_label_range(const float* __restrict__ y, int64_t N, int* __restrict__ bad) {
  int k = 0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < N;
       i += (int64_t)gridDim.x * blockDim.x)
    k += !(y[i] >= 0.0f && y[i] <= 1.0f);
  if (k) atomicAdd(bad, k);
}

// GEMM1's fp32 order: out[T][q][lane][j] = X[32 T + lane % 32][8 q + 2 j + lane / 32],
// four k-steps of a lane in 16 bytes.
__global__ void __launch_bounds__(256)
split_prep_a(const float* __restrict__ X, int64_t N, int D, int Q, int64_t ntile,
             f32x4* __restrict__ out) {
  const int64_t total = ntile * Q * 64;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int lane = (int)(i % 64);
    const int64_t r = i / 64;
    const int q = (int)(r % Q);
    const int64_t n = 32 * (r / Q) + lane % 32;
    f32x4 v;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int d = 8 * q + 2 * j + lane / 32;
      v[j] = (n < N && d < D) ? X[n * D + d] : 0.0f;
    }
    out[i] = v;
  }
}

// GEMM2's fp32 order: out[T][m4][dt][lane][j] = X[32 T + row][32 dt + lane % 32] for
// the accumulator register m = 4 m4 + j, row = 8 m4 + 4 (lane / 32) + j.
__global__ void __launch_bounds__(256)
split_prep_b(const float* __restrict__ X, int64_t N, int D, int DT, int64_t ntile,
             f32x4* __restrict__ out) {
  const int64_t total = ntile * 4 * DT * 64;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int lane = (int)(i % 64);
    int64_t r = i / 64;
    const int dt = (int)(r % DT);
    r /= DT;
    const int m4 = (int)(r % 4);
    const int d = 32 * dt + lane % 32;
    f32x4 v;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t n = 32 * (r / 4) + 8 * m4 + 4 * (lane / 32) + j;
      v[j] = (n < N && d < D) ? X[n * D + d] : 0.0f;
    }
    out[i] = v;
  }
}

// Position of a lane's 8 values in an fp16 fragment block: the second half's
// rows are stored XOR 4, so that the transposed reads of a row's two 8-column
// halves fall on different LDS banks.
__device__ __forceinline__ int frag_lane(int pos) { return pos ^ ((pos >> 5) << 2); }

// fp16 order: out[T][plane][kk][pos][8], value j of lane l = frag_lane(pos) is the hi
// (plane 0) or lo term of X[32 T + l % 32][16 kk + 8 (l / 32) + j] / cscale.
__global__ void __launch_bounds__(256)
split_prep_h(const float* __restrict__ X, int64_t N, int D, int KK, int64_t ntile,
             const float* __restrict__ cscale, const float* __restrict__ cgrid,
             f16x8* __restrict__ out) {
  const int64_t total = ntile * KK * 64;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int pos = (int)(i % 64), lane = frag_lane(pos);
    const int64_t r = i / 64;
    const int kk = (int)(r % KK);
    const int64_t t = r / KK;
    const int64_t n = 32 * t + lane % 32;
    f16x8 hi, lo;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int d = 16 * kk + 8 * (lane / 32) + j;
      _Float16 h, l;
      const bool ok = n < N && d < D;
      split16(ok ? X[n * D + d] / cscale[d] : 0.0f, ok ? cgrid[d] : 1.0f, h, l);
      hi[j] = h;
      lo[j] = l;
    }
    out[((t * 2) * KK + kk) * 64 + pos] = hi;
    out[((t * 2 + 1) * KK + kk) * 64 + pos] = lo;
  }
}

// The same order for e4m3 codes (row-major [N][D]), one byte each; padding is
// code 0 (the value 0).
__global__ void __launch_bounds__(256)
split_prep_fp8(const uint8_t* __restrict__ q, int64_t N, int D, int KK, int64_t ntile,
               uint2* __restrict__ out) {
  const int64_t total = ntile * KK * 64;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int pos = (int)(i % 64), lane = frag_lane(pos);
    const int64_t r = i / 64;
    const int kk = (int)(r % KK);
    const int64_t t = r / KK;
    const int64_t n = 32 * t + lane % 32;
    unsigned w[2] = {0, 0};
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int d = 16 * kk + 8 * (lane / 32) + j;
      const unsigned c = (n < N && d < D) ? q[n * D + d] : 0;
      w[j / 4] |= c << (8 * (j % 4));
    }
    out[i] = uint2{w[0], w[1]};
  }
}

__global__ void split_pad_y(const float* __restrict__ y, int64_t N, int64_t Np,
                            float* __restrict__ out) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < Np;
       i += (int64_t)gridDim.x * blockDim.x)
    out[i] = i < N ? y[i] : 0.5f;
}

// ---- the fused kernel ----------------------------------------------------------------

// kSplitF32: fp32 design, GEMM2 by fp16 terms; kPlainF32: GEMM2 on the fp32
// MFMA; kSplitFp8: e4m3 codes, GEMM2 by fp16 terms of R.
enum { kSplitF32 = 0, kPlainF32 = 1, kSplitFp8 = 2 };

// Bytes of a tile's GEMM1 part (A, fp32) and GEMM2 part (B) in LDS, and the slots
// of their rings.
template <int DP, int MODE>
struct SplitShape {
  static constexpr int KK = DP / 16, DT = DP / 32;
  static constexpr int ABYTES = 128 * DP;
  static constexpr int BBYTES = MODE == kSplitFp8 ? 64 * DP : 128 * DP;
  static constexpr int NS = MODE == kSplitFp8 ? 3 : DP <= 64 ? 4 : DP == 128 || DP > 192 ? 2 : 3;
  static constexpr int NA = MODE == kSplitFp8 ? 2 : NS;
};
// blocks per CU: registers (z and the accumulators) up to 128 columns, two
__host__ __device__ constexpr int split_occ(int dp, int mode) {
  return dp <= 128 && mode != kPlainF32 ? 2 : 1;
}

// The block's row tiles i = 0..n-1 (tile rb + i RB) pass through rings in LDS.
// Iteration i: GEMM1 of tile i + 1 interleaved with the epilogue of tile i,
// then GEMM2 of tile i.  A of tile i + NS and B of tile i + NS - 1 are issued
// into the slots that tiles i and i - 1 left (direct global->LDS loads, waited
// for with a count); fp8: codes of tile i + 3 to registers, tile i + 2 decoded
// into LDS, as fp32 for GEMM1 and as fp16 for GEMM2.
template <int DP, int MODE>
__global__ void __launch_bounds__(256, split_occ(DP, MODE))
logit_split_kernel(const void* __restrict__ XA, const void* __restrict__ XB,
                   const float* __restrict__ cscale, const float* __restrict__ ypad,
                   int64_t N, int64_t ntile, const float* __restrict__ Z, int ldz, int D, int C,
                   float* __restrict__ wsg, double* __restrict__ wsu,
                   const int* __restrict__ act, const int* __restrict__ nact) {
  using SH = SplitShape<DP, MODE>;
  constexpr int KK = SH::KK, DT = SH::DT, NS = SH::NS, NA = SH::NA;
  constexpr int AB = SH::ABYTES, BB = SH::BBYTES, PLANE = KK * 64 * 16;
  constexpr bool FP8 = MODE == kSplitFp8;
  constexpr int STEPS = DP / 2;  // GEMM1 k-steps
  // parts of 8 columns that may lie past D and are then skipped (wider designs
  // lose more by the branches than the parts take)
  constexpr int QSKIP = DP <= 128 ? DP / 8 - 3 : DP / 8;
  __shared__ __attribute__((aligned(16))) char lds_a[NA][AB];
  __shared__ __attribute__((aligned(16))) char lds_b[NS][BB];
  __shared__ __attribute__((aligned(16))) char lds_y[NS][128];

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l = tid & 63;
  const int cl = l & 31, h = l >> 5;
  // Chains are taken through the compacted list act[0..*nact) of the chains
  // that requested a gradient (all C in order when act is null); column
  // index ci addresses the workspaces (row stride CT * 128), chain act[ci]
  // the positions.
  const int n_act = act ? *nact : C;
  if (n_act <= 0) return;
  int CT, RB;
  logit_split(n_act, (int)gridDim.x, ntile, CT, RB);
  const int ldw = CT * 128;
  const int bid = blockIdx.x;
  const int xcd = bid & 7;  // blocks of one row split share an XCD
  const int slot = bid >> 3;
  const int ct = slot % CT;
  const int rb = (slot / CT) * 8 + xcd;
  if (rb >= RB) return;  // uniform over the block
  const int c0 = ct * 128 + wave * 32;
  const bool cvalid = c0 + cl < n_act;
  const int c = cvalid ? (act ? act[c0 + cl] : c0 + cl) : 0;

  // GEMM1's B operand: lane (c, h) holds z[2 k + h] of k-step k (fp8: times the
  // column's scale, exact)
  float zf[STEPS];
  const float* zc = Z + (size_t)c * ldz;
#pragma unroll
  for (int k = 0; k < STEPS; ++k) {
    const int d = 2 * k + h;
    zf[k] = (cvalid && d < D) ? (FP8 ? zc[d] * cscale[d] : zc[d]) : 0.0f;
  }
  f32x16 g[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int v = 0; v < 16; ++v) g[dt][v] = 0.0f;
  CompSum u;  // fp64 energy over this lane's tiles, compensated

  const int64_t n = rb < ntile ? (ntile - 1 - rb) / RB + 1 : 0;
  // tile i clamped to the block's last, so that every load is in bounds and
  // every wave issues the same number in every iteration
  auto tile_of = [&](int64_t i) { return rb + (i < n ? i : n - 1) * (int64_t)RB; };

  // DP / 32 wave-loads of 64 16-byte chunks per part and wave; the 32 labels
  // are 8 chunks, lanes 0-1 of each wave
  constexpr int NLOAD = 2 * (DP / 32) + 1;
  auto issue_part = [&](const void* src, int64_t i, char* dst) {
    const char* s = (const char*)src + (size_t)tile_of(i) * (128 * DP);
#pragma unroll
    for (int p = 0; p < DP / 32; ++p)
      lds_dma16(s + 16 * (tid + 256 * p), lds_addr(dst + 16 * (256 * p + 64 * wave)));
  };
  auto issue_a = [&](int64_t i) { issue_part(XA, i, lds_a[i % NA]); };
  auto issue_b = [&](int64_t i) {
    issue_part(XB, i, lds_b[i % NS]);
    if (l < 2)
      lds_dma16(ypad + 32 * tile_of(i) + 4 * (2 * wave + l), lds_addr(lds_y[i % NS] + 32 * wave));
  };
  // fp8: 16-byte chunks of codes (two fragments each) through registers
  constexpr int NQ = 2 * DP;  // chunks of a tile
  constexpr int PQ = (NQ + 255) / 256;
  u32x4 pq[FP8 ? PQ : 1];
  f32x4 pqy;
  auto load_codes = [&](int64_t i) {
    const int64_t t = tile_of(i);
    const u32x4* src = (const u32x4*)XB + (size_t)t * NQ;
#pragma unroll
    for (int p = 0; p < PQ; ++p)
      if (NQ % 256 == 0 || tid + 256 * p < NQ) pq[p] = src[tid + 256 * p];
    pqy = ((const f32x4*)(ypad + 32 * t))[tid & 7];
  };
  auto decode = [&](int64_t i) {
    const int s = (int)(i % NS);
#pragma unroll
    for (int p = 0; p < PQ; ++p) {
      if (NQ % 256 == 0 || tid + 256 * p < NQ) {
        f16x8* dst = (f16x8*)(lds_b[s] + 32 * (tid + 256 * p));
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          f16x8 v;
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const unsigned w = pq[p][2 * k + j];
            typedef _Float16 h2 __attribute__((ext_vector_type(2)));
            const h2 a = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, 1.0f, false);
            const h2 b = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, 1.0f, true);
            v[4 * j] = a[0];
            v[4 * j + 1] = a[1];
            v[4 * j + 2] = b[0];
            v[4 * j + 3] = b[1];
          }
          dst[k] = v;
          // columns 8 q .. 8 q + 7 of a row: even ones to lane half 0 of A
          const int f = 2 * (tid + 256 * p) + k;
          const int lane = frag_lane(f & 63);
          const int q = 2 * (f >> 6) + (lane >> 5);
          f32x4* da = (f32x4*)lds_a[i % NA] + q * 64 + (lane & 31);
          da[0] = f32x4{(float)v[0], (float)v[2], (float)v[4], (float)v[6]};
          da[32] = f32x4{(float)v[1], (float)v[3], (float)v[5], (float)v[7]};
        }
      }
    }
    ((f32x4*)lds_y[s])[tid & 7] = pqy;  // equal values from every thread
  };

  auto mma32 = [](float a, float b, const f32x16& acc) -> f32x16 {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, acc, 0, 0, 0);
  };
  auto mma16 = [](f16x8 a, f16x8 b, const f32x16& acc) -> f32x16 {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, acc, 0, 0, 0);
  };
  // GEMM1 k-steps 4 q .. 4 q + 3 of a tile (columns 8 q .. 8 q + 7).
  auto part = [&](int64_t i, int q) -> f32x4 {
    return ((const f32x4*)lds_a[i % NA])[q * 64 + l];
  };
  auto gemm1_part = [&](f32x4 a, int q, f32x16& L) {
#pragma unroll
    for (int j = 0; j < 4; ++j) L = mma32(a[j], zf[4 * q + j], L);
  };
  // GEMM2's B operand for the fp16 MFMA (m2, dt): X rows 16 m2 + 8 (j / 4) +
  // 4 h + j % 4 (the K order that makes R^T the GEMM1 accumulator registers),
  // column 32 dt + lane % 32, by two transposed reads of the tile: in each
  // 16-lane group, lane q returns element q % 4 of the 8-byte chunks addressed
  // by lanes q / 4 + 4 k.
  const int jl = l & 15, gl = l >> 4;
  const int hb = (jl & 3) >> 1;
  const int tr_off =
      (((gl & 1) * 64 + hb * 32 + 4 * ((gl >> 1) ^ hb) + (jl >> 2)) * 16) + 8 * (jl & 1);
  auto bfrag = [&](const char* plane, int m2, int dt) -> f16x8 {
    typedef short v4s __attribute__((ext_vector_type(4)));
    const char* base = plane + tr_off + dt * 2048 + m2 * 256;
    const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) v4s*)(base));
    const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) v4s*)(base + 128));
    return __builtin_bit_cast(f16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };

  if (n > 0) {
    if constexpr (FP8) {
      load_codes(0);
      decode(0);
      load_codes(1);
      decode(1);
      load_codes(2);
    } else {
#pragma unroll 1
      for (int i = 0; i < NS; ++i) issue_a(i);
#pragma unroll 1
      for (int i = 0; i < NS - 1; ++i) issue_b(i);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    __syncthreads();
    f32x16 Lc;
#pragma unroll
    for (int v = 0; v < 16; ++v) Lc[v] = 0.0f;
#pragma unroll
    for (int q = 0; q < DP / 8; ++q)
      if (q < QSKIP || 8 * q < D) gemm1_part(part(0, q), q, Lc);
    __syncthreads();  // A's slot of tile 0 is refilled next
    for (int64_t i = 0; i < n; ++i) {
      if constexpr (FP8) {
        decode(i + 2);
        load_codes(i + 3);
      } else {
        issue_a(i + NS);
        issue_b(i + NS - 1);
      }
      const char* cur = lds_b[i % NS];
      float yv[16];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4 yq = *(const f32x4*)(lds_y[i % NS] + 4 * (8 * q + 4 * h));
#pragma unroll
        for (int m = 0; m < 4; ++m) yv[4 * q + m] = yq[m];
      }
      f32x16 Ln;
#pragma unroll
      for (int v = 0; v < 16; ++v) Ln[v] = 0.0f;
      f16x8 ra[2], rm[2], rc[2];  // R' = ra + (rm + rc) / kRFine
      float rv[16];
      float us = 0.0f;
      f32x4 w = part(i + 1, 0);
      // Rows past N have X = 0 and y = 1/2, so r = 0 exactly and u = fp32(ln 2)
      // (removed below or by the reduction); chains past C have Z = 0 and are
      // never written.  GEMM1 of tile i + 1 (the last tile again at the end) takes
      // turns with the epilogue of tile i, element by element; its LDS reads run
      // one part ahead (scheduling barriers keep them and the VALU work in the
      // MFMAs' shadow).
#pragma unroll
      for (int e = 0; e < 16; ++e) {
#pragma unroll
        for (int q = e * (DP / 8) / 16; q < (e + 1) * (DP / 8) / 16; ++q)
        {
          const f32x4 wn = part(i + 1, q + 1 < DP / 8 ? q + 1 : q);
          if (q < QSKIP || 8 * q < D) gemm1_part(w, q, Ln);
          w = wn;
        }
        float r, uu;
        if constexpr (FP8) logit_terms_log1p(Lc[e], yv[e], r, uu);
        else logit_terms(Lc[e], yv[e], r, uu);
        if constexpr (FP8) {
          u.add((double)uu);
        } else {
          us += uu;
          asm volatile("" : "+v"(us));  // keeps this element's loss term in place
        }
        if constexpr (MODE == kPlainF32) {
          rv[e] = r;
        } else {
          const float v = r * kRScale;
          constexpr float m = 12582912.0f * kRGrid;  // rounds to the grid
          const float hi = (v + m) - m;
          const float rest = (v - hi) * kRFine;  // exact
          const _Float16 mid = (_Float16)rest;
          ra[e / 8][e % 8] = (_Float16)hi;
          rm[e / 8][e % 8] = mid;
          rc[e / 8][e % 8] = (_Float16)(rest - (float)mid);
        }
        if (e < 15) __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (MODE == kPlainF32) {
        // a partial last tile: the sum again without the rows past N, which on
        // designs of a few rows would round off the others' bits
        if (tile_of(i) == ntile - 1 && 32 * ntile > N) {
          us = 0.0f;
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            float r, uu;
            logit_terms(Lc[e], yv[e], r, uu);
            if (32 * (ntile - 1) + 8 * (e / 4) + 4 * h + e % 4 < N) us += uu;
          }
        }
      }
      if constexpr (!FP8) u.add((double)us);
      Lc = Ln;
      if constexpr (MODE == kPlainF32) {
#pragma unroll
        for (int m4 = 0; m4 < 4; ++m4)
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) {
            const f32x4 b = ((const f32x4*)cur)[(m4 * DT + dt) * 64 + l];
#pragma unroll
            for (int j = 0; j < 4; ++j) g[dt] = mma32(rv[4 * m4 + j], b[j], g[dt]);
          }
      } else {
        // column block dt: products of R's grid terms to g, of its fine terms to t
        // from zero; after(k) follows product k
        constexpr int NP = FP8 ? 6 : 10;
        auto products = [&](int dt, f32x16& t, auto after) {
#pragma unroll
          for (int v = 0; v < 16; ++v) t[v] = 0.0f;
#pragma unroll
          for (int m2 = 0; m2 < 2; ++m2) {
            int k = m2 * (NP / 2);
            const f16x8 bh = bfrag(cur, m2, dt);
            f16x8 bl;
            if constexpr (!FP8) bl = bfrag(cur + PLANE, m2, dt);
            t = mma16(rc[m2], bh, t);
            after(k++);
            if constexpr (!FP8) {
              g[dt] = mma16(ra[m2], bl, g[dt]);
              after(k++);
              t = mma16(rm[m2], bl, t);
              after(k++);
            }
            g[dt] = mma16(ra[m2], bh, g[dt]);
            after(k++);
            t = mma16(rm[m2], bh, t);
            after(k++);
          }
        };
        auto fold = [&](int dt, const f32x16& t, int v0, int v1) {
#pragma unroll
          for (int v = v0; v < v1; ++v) g[dt][v] = fmaf(t[v], 1.0f / kRFine, g[dt][v]);
        };
        if constexpr (split_occ(DP, MODE) > 1) {
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) {
            f32x16 t;
            products(dt, t, [](int) {});
            fold(dt, t, 0, 16);
          }
        } else {
          // one wave per SIMD: a block's fine sums are added between the
          // products of the next one
          f32x16 t[2];
#pragma unroll
          for (int dt = 0; dt < DT; ++dt)
            products(dt, t[dt & 1], [&](int k) {
              if (dt > 0) fold(dt - 1, t[(dt - 1) & 1], 16 * k / NP, 16 * (k + 1) / NP);
              __builtin_amdgcn_sched_barrier(0);
            });
          fold(DT - 1, t[(DT - 1) & 1], 0, 16);
        }
      }
      if constexpr (!FP8) {
        // A of tile i + 2 and B of tile i + 1 must be there for the next
        // iteration; what later iterations need may still be in flight (loads
        // retire in order)
        static_assert((NS - 2) * NLOAD < 64, "vmcnt holds 6 bits");
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 2) * NLOAD) : "memory");
      }
      __syncthreads();
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }

#pragma unroll
  for (int dt = 0; dt < DT; ++dt) {
    const int d = 32 * dt + cl;
    if (d < D) {
      const float sc = MODE == kPlainF32 ? 1.0f : cscale[d] / kRScale;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int ci = c0 + 8 * (v / 4) + 4 * h + (v % 4);
        if (ci < n_act) wsg[((size_t)rb * ldw + ci) * D + d] = g[dt][v] * sc;
      }
    }
  }
  CompSum uo;
  uo.s = __shfl_xor(u.s, 32, 64);
  uo.c = __shfl_xor(u.c, 32, 64);
  u.add(uo);
  const double ut = u.value();
  if (h == 0 && cvalid) wsu[(size_t)rb * ldw + c0 + cl] = ut;
}

struct LogisticSplit : Potential {
  int64_t n = 0, ntile = 0;
  int d = 0, dp = 0;
  double prior_scale = 1.0;
  int mode = kSplitF32;
  void* xa = nullptr;
  void* xb = nullptr;
  float* cscale = nullptr;  // [d], and for the split the columns' grids [d]
  float* ypad = nullptr;
  float* wsg = nullptr;
  double* wsu = nullptr;
  size_t ws_elems = 0;
  int num_cu = 256;

  ~LogisticSplit() override {
    (void)hipFree(xa);
    (void)hipFree(xb);
    (void)hipFree(cscale);
    (void)hipFree(ypad);
    (void)hipFree(wsg);
    (void)hipFree(wsu);
  }
  int dim() const override { return d; }
  const char* name() const override {
    return mode == kSplitFp8 ? "logit_split_fp8"
                             : (mode == kSplitF32 ? "logit_split_f32" : "logit_mfma_f32");
  }
  double alg_flops(int C) const override { return 4.0 * (double)n * d * C; }
  double alg_bytes(int) const override {
    return (mode == kSplitFp8 ? 1.0 : 4.0) * (double)n * d + 4.0 * n;
  }

  // Row splits of a launch over C chains: one or two 4-wave blocks per CU,
  // a multiple of the 8 XCDs; fp8: at most kSplitRows rows each.
  int row_splits(int C) const {
    const int CT = (C + 127) / 128;
    int64_t RB = std::max(8, (num_cu * split_occ(dp, mode) / CT) / 8 * 8);
    if (mode == kSplitFp8) RB = std::max<int64_t>(RB, (n / kSplitRows + 8) / 8 * 8);
    return (int)std::min<int64_t>(RB, (ntile + 7) / 8 * 8);
  }

  // The split of GEMM2 takes the design (fp32): the range rules of the header.
  hipError_t column_scales(const float* x, const float* y, hipStream_t s, bool* ok) {
    char* tmp = nullptr;  // [blocks][d] doubles, then bits, then the count
    const size_t cells = (size_t)kStatBlocks * d;
    hipError_t e = hipMallocAsync((void**)&tmp, cells * 12 + sizeof(int), s);
    if (e != hipSuccess) return e;
    double* psq = reinterpret_cast<double*>(tmp);
    unsigned* pmax = reinterpret_cast<unsigned*>(tmp + cells * 8);
    int* bad = reinterpret_cast<int*>(tmp + cells * 12);
    int hbad = 0;
    e = hipMemsetAsync(bad, 0, sizeof(int), s);
    if (e == hipSuccess) {
      hipLaunchKernelGGL(split_col_stats, dim3(kStatBlocks), dim3(256), 0, s, x, n, d, pmax, psq);
      hipLaunchKernelGGL(split_col_scale, dim3(1), dim3(256), 0, s, pmax, psq, kStatBlocks, n, d,
                         cscale, cscale + d, bad);
      hipLaunchKernelGGL(split_label_range, dim3(256), dim3(256), 0, s, y, n, bad);
      e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpyAsync(&hbad, bad, sizeof(int), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    (void)hipFreeAsync(tmp, s);
    *ok = hbad == 0;
    return e;
  }

  // X fp32 row-major, or its codes and column scales (fp8).
  hipError_t setup(const float* x, const uint8_t* codes, const float* scales, const float* y,
                   int num_chains, bool fp32_products, hipStream_t s) {
    ntile = (n + 31) / 32;
    dp = (d + 31) / 32 * 32;
    int dev = 0;
    hipDeviceProp_t prop;
    if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess)
      num_cu = prop.multiProcessorCount;
    hipError_t e = hipMalloc(&cscale, sizeof(float) * 2 * d);
    if (e != hipSuccess) return e;
    if (codes) {
      mode = kSplitFp8;
      e = hipMemcpyAsync(cscale, scales, sizeof(float) * d, hipMemcpyDeviceToDevice, s);
    } else {
      mode = kSplitF32;
      bool ok = !fp32_products && n >= kSplitMin && n <= kSplitRows * row_splits(num_chains);
      if (ok) e = column_scales(x, y, s, &ok);
      if (!ok) mode = kPlainF32;
    }
    if (e != hipSuccess) return e;
    const size_t elems = (size_t)ntile * 32 * dp;
    if (mode != kSplitFp8) e = hipMalloc(&xa, elems * 4);
    if (e == hipSuccess) e = hipMalloc(&xb, elems * (mode == kSplitFp8 ? 1 : 4));
    if (e == hipSuccess) e = hipMalloc(&ypad, sizeof(float) * ntile * 32);
    if (e != hipSuccess) return e;
    const dim3 gr(4096), bl(256);
    if (mode == kSplitFp8)
      hipLaunchKernelGGL(split_prep_fp8, gr, bl, 0, s, codes, n, d, dp / 16, ntile, (uint2*)xb);
    else
      hipLaunchKernelGGL(split_prep_a, gr, bl, 0, s, x, n, d, dp / 8, ntile, (f32x4*)xa);
    if (mode == kSplitF32)
      hipLaunchKernelGGL(split_prep_h, gr, bl, 0, s, x, n, d, dp / 16, ntile, cscale,
                         cscale + d, (f16x8*)xb);
    else if (mode == kPlainF32)
      hipLaunchKernelGGL(split_prep_b, gr, bl, 0, s, x, n, d, dp / 32, ntile, (f32x4*)xb);
    hipLaunchKernelGGL(split_pad_y, dim3(1024), bl, 0, s, y, n, ntile * 32, ypad);
    e = hipGetLastError();
    return e != hipSuccess ? e : hipStreamSynchronize(s);
  }

  hipError_t eval(hipStream_t s, const float* z, int ldz, int C, double* pe, float* g,
                  int ldg) override {
    return eval_active(s, z, ldz, C, nullptr, nullptr, pe, g, ldg);
  }
  hipError_t eval_active(hipStream_t s, const float* z, int ldz, int C, const int* act,
                         const int* nact, double* pe, float* g, int ldg) override {
    const int RB = row_splits(C);
    const int nblk = (C + 127) / 128 * RB;
    // the kernels re-split the launch for the requesting chains: RB' CT' <=
    // nblk, row stride CT' 128, so nblk * 128 columns always suffice
    const size_t need = (size_t)nblk * 128 * d;
    if (need > ws_elems) {
      (void)hipFree(wsg);
      (void)hipFree(wsu);
      wsg = nullptr;
      wsu = nullptr;
      ws_elems = 0;
      hipError_t e = hipMalloc(&wsg, sizeof(float) * need);
      if (e != hipSuccess) return e;
      e = hipMalloc(&wsu, sizeof(double) * (size_t)nblk * 128);
      if (e != hipSuccess) return e;
      ws_elems = need;
    }
    mark_begin(s);
#define NAX_S(DPV, MD)                                                                          \
  case DPV:                                                                                     \
    hipLaunchKernelGGL((logit_split_kernel<DPV, MD>), dim3(nblk), dim3(256), 0, s, xa, xb,       \
                       cscale, ypad, n, ntile, z, ldz, d, C, wsg, wsu, act, nact);              \
    break;
#define NAX_SDP(MD)                                                                             \
  switch (dp) {                                                                                 \
    NAX_S(32, MD) NAX_S(64, MD) NAX_S(96, MD) NAX_S(128, MD)                                    \
    NAX_S(160, MD) NAX_S(192, MD) NAX_S(224, MD) NAX_S(256, MD)                                 \
    default: return hipErrorInvalidValue;                                                       \
  }
    if (mode == kSplitFp8) {
      NAX_SDP(kSplitFp8)
    } else if (mode == kSplitF32) {
      NAX_SDP(kSplitF32)
    } else {
      NAX_SDP(kPlainF32)
    }
#undef NAX_SDP
#undef NAX_S
    mark_end(s);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const double inv_s2 = 1.0 / (prior_scale * prior_scale);
    const double log_norm = std::log(std::sqrt(2.0 * M_PI) * prior_scale);
    // padded rows each added fp32(ln 2) to every chain's energy (split forms)
    const float pad = mode == kSplitFp8 ? log1pf(1.0f) : 0.693147180559945309f;
    const double pad_u = mode == kPlainF32 ? 0.0 : (double)(ntile * 32 - n) * (double)pad;
    hipLaunchKernelGGL(logit_reduce, dim3(C), dim3(reduce_threads(C)), 0, s, wsg, wsu, RB, C, d, z, ldz, inv_s2,
                       log_norm, -pad_u, pe, g, ldg, act, nact, nblk, ntile);
    return hipGetLastError();
  }
};

int64_t logistic_split_min_rows() { return kSplitMin; }

// Whether every label is in [0, 1], as the forms in fp16 terms need it.
hipError_t logistic_split_labels(const float* y, int64_t n, hipStream_t s, bool* ok) {
  int* bad = nullptr;
  int hbad = 0;
  hipError_t e = hipMallocAsync((void**)&bad, sizeof(int), s);
  if (e != hipSuccess) return e;
  e = hipMemsetAsync(bad, 0, sizeof(int), s);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(split_label_range, dim3(256), dim3(256), 0, s, y, n, bad);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipMemcpyAsync(&hbad, bad, sizeof(int), hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  (void)hipFreeAsync(bad, s);
  *ok = hbad == 0;
  return e;
}

// fp32 X, or (codes given) its e4m3 codes [n][d] and column scales [d], which
// are copied; d <= 256, n rows for num_chains chains.  fp32_products: X^T R on the
// fp32 MFMA whatever the design.
Potential* make_logistic_split(const float* x, const uint8_t* codes, const float* scales,
                               const float* y, int64_t n, int d, double prior_scale,
                               int num_chains, bool fp32_products, hipStream_t s,
                               std::string* err) {
  if (d > 256) {
    *err = "the MFMA logistic kernels support dim <= 256";
    return nullptr;
  }
  auto* p = new LogisticSplit();
  p->n = n;
  p->d = d;
  p->prior_scale = prior_scale;
  const hipError_t e = p->setup(x, codes, scales, y, num_chains, fp32_products, s);
  if (e != hipSuccess) {
    *err = std::string("logistic matrix-core setup: ") + hipGetErrorString(e);
    delete p;
    return nullptr;
  }
  return p;
}

}  // namespace nax
