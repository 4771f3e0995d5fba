// Many independent non-centred hierarchical logistic regressions of uneven
// size, K chains per model, in one launch.
//
// Model i (rows N_i, columns D_i <= 64):
//   eta ~ Normal(0, 1)^D_i, mu ~ Normal(0, 1), tau ~ HalfCauchy(1),
//   beta = mu + tau * eta, y_n ~ Bernoulli(logits = x_n . beta)
// (Normal continuous.py:2975-2989, HalfCauchy continuous.py:1149-1150 ->
// Cauchy continuous.py:390-406, BernoulliLogits discrete.py:244-263; tau is
// unconstrained by ExpTransform, transforms.py:606-652, log|J| = log tau).
// Latent of a chain, sorted site names: [eta (D_i), mu, log tau].
//
// Data are ragged row-major blocks: X rows of model i at elt_off[i], labels at
// row_off[i].  A block of K wavefronts owns model i and its K chains: one X
// tile of 64 rows is staged in LDS once and used by all K chains (phase 1:
// lane = row, wave = chain -> logits and residuals; phase 2: lane = column,
// wave = chain -> X^T R), so each byte of X_i is read once per gradient tick
// of the model, not once per chain.  In the persistent form each wave runs
// its chain's NUTS state machine; when any chain of the block needs a
// gradient the block evaluates all K together (chains that are already done
// ride along and ignore the result).  Blocks take models heaviest first
// (N_i D_i descending) to even out the tail of the launch.  A model's K
// chains may also be split over K / KB workgroups of KB chains each (each
// then reads X_i for its KB chains): more workgroups for the heavy models
// against more passes over their X.  And each chain may own R waves: the
// block then stages R tiles (64 R rows) at a time, wave r of a chain takes
// rows 64 r .. 64 r + 63 of them in both phases, and the R partial sums of
// U and X^T R are added in r order at the end -- a heavy model's leaf then
// takes ~1/R of the time, which is what the launch waits for.  The NUTS
// state machine of a chain runs on its wave r = 0.  The autotuner picks
// (KB, R).  One evaluation outside a run, where no chain waits for another, has a
// kernel of its own (hier_once_kernel).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <numeric>
#include <string>
#include <vector>

#include "nax_device.h"
#include "nax_engine.h"
#include "nax_internal.h"

namespace nax {

constexpr int kHierRows = 64;
constexpr int kHierMaxD = 64;
constexpr double kLog2PiHalf = 0.91893853320467274;
constexpr double kLogPi_ = 1.1447298858494002;
constexpr double kLog2 = 0.69314718055994531;

struct HierData {
  const float* x;
  const float* y;
  const int64_t* row_off;
  const int64_t* elt_off;
  const int* dims;
  const int* order;  // block -> model, heaviest first
  int K;             // chains per model
  int Dp;            // stride of a chain's latent vector
  int softplus;      // tau by SoftplusTransform instead of ExpTransform
};

// Row stride of a staged X tile: 68 floats keeps both access patterns free
// of LDS bank conflicts (lane = row reading 16-byte column groups, lane =
// column reading one row) and 16-byte aligned.
constexpr int kHierLd = kHierMaxD + 4;

template <int K, int R>
struct __attribute__((aligned(16))) HierShared {
  __attribute__((aligned(16))) float xs[2][kHierRows * R][kHierLd];  // double-buffered X tiles
  __attribute__((aligned(16))) float beta[K][kHierMaxD];
  __attribute__((aligned(16))) float res[K][kHierRows * R];  // residuals sigmoid(l) - y, chain-major
  float ys[2][kHierRows * R];
  // partial X^T R and U of the R waves of each chain (R > 1)
  __attribute__((aligned(16))) float racc[R > 1 ? K : 1][R > 1 ? R : 1][kHierMaxD];
  double rul[R > 1 ? K : 1][R > 1 ? R : 1];
};

// Tiles held in registers ahead of the one being processed: enough bytes in
// flight per workgroup to cover the memory latency when a model's workgroup
// runs alone on its CU (the tail of a launch), within ~64 VGPRs.
template <int K, int R>
struct HierPipe {
  static constexpr int NT = 64 * K * R;                       // threads
  static constexpr int EPT = kHierRows * R * kHierMaxD / NT;  // tile elements per thread
  static constexpr int PF = (EPT >= 32) ? 1 : 2;
};

// U and dU of a chain at z from its likelihood part U_lik and, lane = column,
// the column's X^T r (0 past D), on one wave.
__device__ inline double hier_finish(const HierData& hd, int D, int lane, const float* z, float acc,
                                     double U_lik, float* g) {
  const float mu = z[D];
  const PosTf tt = positive_tf((double)z[D + 1], hd.softplus != 0);
  const float tau = hd.softplus ? (float)tt.x : expf(z[D + 1]);
  const float eta = lane < D ? z[lane] : 0.0f;
  // dU/deta = eta + tau acc, dU/dmu = mu + sum acc,
  // dU/dlog tau = tau eta.acc + 2 tau^2 / (1 + tau^2) - 1
  const double sum_acc = wave_sum((double)acc);
  const double eta_acc = wave_sum((double)eta * acc);
  const double eta2 = wave_sum((double)eta * eta);
  if (lane < D) g[lane] = eta + tau * acc;
  const double t2 = (double)tau * tau;
  if (lane == 0) {
    g[D] = (float)((double)mu + sum_acc);
    // softplus: dtau/du (eta.acc + 2 tau / (1 + tau^2)) - d log|J| / du
    g[D + 1] = hd.softplus
        ? (float)(tt.dx * (eta_acc + 2.0 * (double)tau / (1.0 + t2)) - tt.dladj)
        : (float)((double)tau * eta_acc + 2.0 * t2 / (1.0 + t2) - 1.0);
  }
  const double U = U_lik + 0.5 * eta2 + D * kLog2PiHalf          // eta ~ N(0,1)
                   + 0.5 * (double)mu * mu + kLog2PiHalf          // mu ~ N(0,1)
                   - (kLog2 - kLogPi_ - log1p(t2))                // HalfCauchy(1)
                   - (hd.softplus ? tt.ladj : (double)z[D + 1]);  // log|J|
  return U;
}

// Block-cooperative U and dU for the K chains of model i at z[c] (c = chain
// index of the block's chain slot w: c = i K_model + sub K + w), each chain
// on R waves (wave index w R + r).  Wave r = 0 of slot w ends with its own
// chain's results: returns U on every lane of that wave (0 on the others),
// writes dU to g[c].  Tiles of 64 R rows are contiguous (rows * D floats) in
// the ragged layout.  Tile t is loaded into registers PF tiles ahead, staged
// into LDS buffer t & 1, then: phase 1 (lane = row 64 r + lane, wave =
// chain part) logits and residuals, phase 2 (lane = column, same wave) X^T R
// over the same 64 rows.  One barrier per tile: the residuals a wave writes
// in phase 1 are read back only by that wave (LDS accesses of one wavefront
// complete in order), and buffer t & 1 is next written (tile t + 2) after
// every wave has passed the barrier of tile t + 1.  With R > 1 the R
// partial sums of X^T R and of U are added in r order after the last tile.
template <int K, int R>
__device__ double hier_group_eval(const HierData& hd, int i, int sub, const float* zreq,
                                  int ldz, float* gout, int ldg, HierShared<K, R>& sh) {
  using P = HierPipe<K, R>;
  constexpr int NT = P::NT, EPT = P::EPT, PF = P::PF;
  constexpr int TR = kHierRows * R;  // rows of a staged tile
  const int wa = threadIdx.x >> 6;
  const int w = wa / R;               // chain slot
  const int r = wa % R;               // 64-row part of the tile
  const int lane = threadIdx.x & 63;
  const int D = hd.dims[i];
  const int D4 = (D + 3) & ~3;
  const int64_t N = hd.row_off[i + 1] - hd.row_off[i];
  const int ntiles = (int)((N + TR - 1) / TR);
  const float* X = hd.x + hd.elt_off[i];
  const float* Y = hd.y + hd.row_off[i];
  const int c = i * hd.K + sub * K + w;
  const float* z = zreq + (size_t)c * ldz;
  float* g = gout + (size_t)c * ldg;
  if (r == 0) {
    const float tau = hd.softplus ? (float)positive_tf((double)z[D + 1], true).x : expf(z[D + 1]);
    sh.beta[w][lane] = lane < D ? z[D] + tau * z[lane] : 0.0f;
  }
  // columns [D, D4) of both buffers stay zero for the whole evaluation
  for (int e = threadIdx.x; e < 2 * TR * 4; e += NT) {
    const int b = e / (TR * 4), rr = (e / 4) % TR, cc = D + (e & 3);
    if (cc < D4) sh.xs[b][rr][cc] = 0.0f;
  }
  // element e = threadIdx.x + NT j of a tile sits at row e / D, column e % D
  const int step_r = NT / D, step_c = NT % D;
  const int r_first = threadIdx.x / D, c_first = threadIdx.x % D;
  float px[PF][EPT];
  float py[PF];
  auto load = [&](int t, float* dst, float& ydst) {
    const int64_t r0 = (int64_t)t * TR;
    const int rows = (int)min<int64_t>(TR, N - r0);
    const int ne = rows * D;
    const float* src = X + r0 * D;
#pragma unroll
    for (int j = 0; j < EPT; ++j) {
      const int e = threadIdx.x + NT * j;
      dst[j] = e < ne ? src[e] : 0.0f;
    }
    ydst = threadIdx.x < rows ? Y[r0 + threadIdx.x] : 0.0f;
  };
#pragma unroll
  for (int j = 0; j < PF; ++j)
    if (j < ntiles) load(j, px[j], py[j]);
  const int rr0 = kHierRows * r;  // this wave's first row in a tile
  float acc = 0.0f;   // phase 2: dU/dbeta_lane for chain w over this wave's rows
  double ul = 0.0;    // phase 1: likelihood part of U for chain w over this wave's rows
  for (int t0 = 0; t0 < ntiles; t0 += PF) {
#pragma unroll
    for (int j = 0; j < PF; ++j) {
      const int t = t0 + j;
      if (t < ntiles) {
        const int rows = (int)min<int64_t>(TR, N - (int64_t)t * TR);
        float(*xs)[kHierLd] = sh.xs[t & 1];
        {
          // the whole tile is written: rows past `rows` get zeros
          const int ne = TR * D;
          int rr = r_first, cc = c_first;
#pragma unroll
          for (int q = 0; q < EPT; ++q) {
            if (threadIdx.x + NT * q < ne) xs[rr][cc] = px[j][q];
            rr += step_r;
            cc += step_c;
            if (cc >= D) { cc -= D; rr += 1; }
          }
          if (threadIdx.x < TR) sh.ys[t & 1][threadIdx.x] = py[j];
        }
        if (t + PF < ntiles) load(t + PF, px[j], py[j]);  // in flight during the compute below
        __syncthreads();
        const int rows_r = min(max(rows - rr0, 0), kHierRows);
        float rv = 0.0f;
        if (lane < rows_r) {
          float l0 = 0.0f, l1 = 0.0f, l2 = 0.0f, l3 = 0.0f;
          const float4* xr = reinterpret_cast<const float4*>(&xs[rr0 + lane][0]);
          const float4* br = reinterpret_cast<const float4*>(&sh.beta[w][0]);
#pragma unroll
          for (int q = 0; q < kHierMaxD / 4; ++q) {
            if (4 * q < D4) {
              const float4 xv = xr[q], bv = br[q];
              l0 = fmaf(xv.x, bv.x, l0);
              l1 = fmaf(xv.y, bv.y, l1);
              l2 = fmaf(xv.z, bv.z, l2);
              l3 = fmaf(xv.w, bv.w, l3);
            }
          }
          float u;
          logistic_terms_f((l0 + l1) + (l2 + l3), sh.ys[t & 1][rr0 + lane], rv, u);
          ul += (double)u;
        }
        sh.res[w][rr0 + lane] = rv;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (lane < D) {
          const int rows4 = (rows_r + 3) & ~3;  // residuals of rows past `rows` are 0
          const float4* rq = reinterpret_cast<const float4*>(&sh.res[w][rr0]);
          float a0 = 0.0f, a1 = 0.0f;
          for (int q = 0; q < rows4 / 4; ++q) {
            const float4 rv4 = rq[q];
            a0 = fmaf(xs[rr0 + 4 * q][lane], rv4.x, a0);
            a1 = fmaf(xs[rr0 + 4 * q + 1][lane], rv4.y, a1);
            a0 = fmaf(xs[rr0 + 4 * q + 2][lane], rv4.z, a0);
            a1 = fmaf(xs[rr0 + 4 * q + 3][lane], rv4.w, a1);
          }
          acc += a0 + a1;
        }
      }
    }
  }
  double U_lik;
  if constexpr (R > 1) {
    sh.racc[w][r][lane] = acc;
    const double uw = wave_sum(ul);
    if (lane == 0) sh.rul[w][r] = uw;
    __syncthreads();
    if (r != 0) return 0.0;
    float a = 0.0f;
    double us = 0.0;
#pragma unroll
    for (int q = 0; q < R; ++q) {
      a += sh.racc[w][q][lane];
      us += sh.rul[w][q];
    }
    acc = a;
    U_lik = us;
  } else {
    U_lik = wave_sum(ul);
  }
  return hier_finish(hd, D, lane, z, acc, U_lik, g);
}

template <int K, int R>
__global__ void __launch_bounds__(64 * K * R)
hier_eval_kernel(HierData hd, const float* __restrict__ zreq, int ldz, double* __restrict__ pe,
                 float* __restrict__ gout, int ldg) {
  __shared__ HierShared<K, R> sh;
  const int per = hd.K / K;  // workgroups per model
  const int i = hd.order[blockIdx.x / per];
  const int sub = blockIdx.x % per;
  const double u = hier_group_eval<K, R>(hd, i, sub, zreq, ldz, gout, ldg, sh);
  const int wa = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0 && wa % R == 0) pe[i * hd.K + sub * K + wa / R] = u;
}

// fourth word of a buffer descriptor: plain 32-bit data
constexpr int kBufferWord3 = 0x00027000;

typedef float f32x4 __attribute__((ext_vector_type(4)));

// One-shot evaluation: waves of a block and rows of a wave's tile (1024 models x
// 4 chains, models whole: 8 x 32 116 us a pass, 4 x 64 130 us; in an earlier
// form 16 x 16 166, 8 x 16 152, 8 x 32 136, 4 x 64 160, 4 x 32 167, 2 x 64 218).
constexpr int kOnceWaves = 8, kOnceRows = 32;
static_assert(kOnceRows % 32 == 0 && kOnceRows <= 64, "tile layout");
// A model above 1 / 256 of all elements (one CU's part) is split into items: 1024
// models of up to 5000 x 64 are then whole, where items of half and of an eighth of
// that cost 6 and 15 us of starting blocks and combining (116 us a pass), and 60
// models x 4 chains still fill the chip (345 -> 112 us a pass).  No item is split
// below 64 KB, two rounds of a block's tiles.
constexpr double kOnceItems = 256.0, kOnceItemMin = 16384.0;

// Rows [row0, row0 + rows) of a model; slot: where the partial sums go, -1 when
// the item is its whole model.
struct HierItem {
  int64_t row0, rows;
  int model, slot;
};
// A model of several items and its first slot.
struct HierSplit {
  int model, slot, count;
};

// U and dU of the K chains of one item's rows, once: the rows in tiles of TR over
// W waves, each wave evaluating all K chains on its tiles, so X_i is read
// once and a tile's bytes leave LDS once for each product instead of once per
// chain.  The tiles are the wave's own (no barrier in the loop): loaded into
// registers one tile ahead, stored into LDS, then
//   logits     lane = row: one v_mfma_f32_4x4x1 (16 blocks of 4 rows x 4 chains)
//              per column and 4 chains: the same four interleaved sums of fused
//              multiply-adds as hier_group_eval, bit for bit
//   residuals  lane = (4 rows, chain) of those accumulators
//   X^T R      lane = column: one v_mfma_f32_4x4x1 per row and 4 chains
// and the waves' partial sums are added in wave order.  Bound: the reads of X and,
// in a block, the start of its first tiles and the finish of its chains (1024
// models x 4 chains, 350 MB: 220 us with a wave per chain on a shared tile, every
// chain reading the tile from LDS and one tile of dword loads in flight; 98 us
// now, against 75 us for a copy of as many bytes).
template <int K, int W, int TR>
__global__ void __launch_bounds__(64 * W, 2)
hier_once_kernel(HierData hd, const HierItem* __restrict__ items, const float* __restrict__ zreq,
                 int ldz, double* __restrict__ pe, float* __restrict__ gout, int ldg,
                 float* __restrict__ part_g, double* __restrict__ part_u) {
  constexpr int SETS = (K + 3) / 4;     // groups of 4 chains
  constexpr int SG = SETS < 2 ? 1 : 2;  // sets at a time: 16 SG accumulator registers
  constexpr int NC = 4 * SETS;
  constexpr int NLD = TR * kHierMaxD / 256;
  // each wave's X tile, at the end its partial X^T R ([chain][column])
  __shared__ __attribute__((aligned(16))) float xs_all[W][TR * kHierLd];
  __shared__ __attribute__((aligned(16))) float beta[NC][kHierLd];  // unused chains: 0
  __shared__ __attribute__((aligned(16))) float res[W][NC][TR + 4];   // sigmoid(l) - y
  __shared__ __attribute__((aligned(16))) float ys[W][TR];
  __shared__ double rul[W][NC];                                       // partial U
  const HierItem it = items[blockIdx.x];
  const int i = it.model;
  const int wa = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int lane = threadIdx.x & 63;
  const int D = hd.dims[i];
  const int64_t N = it.rows;
  const int ntiles = (int)((N + TR - 1) / TR);
  const float* X = hd.x + hd.elt_off[i] + it.row0 * D;
  const float* Y = hd.y + hd.row_off[i] + it.row0;
  for (int q = wa; q < NC; q += W) {
    float b = 0.0f;
    if (q < K && lane < D) {
      const float* z = zreq + (size_t)(i * K + q) * ldz;
      const float tau = hd.softplus ? (float)positive_tf((double)z[D + 1], true).x : expf(z[D + 1]);
      b = z[D] + tau * z[lane];
    }
    beta[q][lane] = b;
  }
  // The wave's own tile.  Its TR D elements are contiguous in memory: loaded and
  // stored to LDS 16 bytes a lane, chunk lane + 64 j of the tile.  Rows are SD
  // apart in LDS: D a multiple of 8 takes 4 floats of padding, which spreads the
  // rows over the banks; any other D is conflict-free (or 2-way) as it is.
  float* xs = xs_all[wa];
  const bool quad = (D & 3) == 0;
  const int SD = (D & 7) == 0 ? D + 4 : D;
  const int nld = (TR * D + 255) / 256;  // 16-byte loads of a tile
  int dst[NLD];
#pragma unroll
  for (int j = 0; j < NLD; ++j) {
    const int e = 4 * (lane + 64 * j);
    dst[j] = SD == D ? e : e + 4 * (e / D);
  }
  f32x4 px[NLD];
  float py = 0.0f;
  const int full = (int)(N / TR);  // tiles of TR rows; at most one more, of fewer
  // Every load of a full tile is issued, without a branch: what lies past the
  // tile's TR D elements (16 bytes never straddle that end) or past the last full
  // tile reads as 0 and takes no memory access.
  auto load = [&](int t) {
    const int64_t r0 = (int64_t)t * TR;
    const int ok = t < full ? 4 * TR : 0;
    const auto rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(X + r0 * D), 0, ok * D,
                                                      kBufferWord3);
    const auto ry =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(Y + r0), 0, ok, kBufferWord3);
#pragma unroll
    for (int j = 0; j < NLD; ++j)
      px[j] = __builtin_bit_cast(
          f32x4, __builtin_amdgcn_raw_buffer_load_b128(rx, 16 * (lane + 64 * j), 0, 0));
    py = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(ry, 4 * lane, 0, 0));
  };
  load(wa);
  const int j4 = lane & 3, b4 = lane >> 2;  // chain of a set, block of 4 rows / columns
  constexpr int RV = TR / 16;  // rows a lane takes the residuals of
  const bool upper = lane >= TR;
  const int rl = 4 * b4 % TR + (upper ? RV : 0);
  f32x4 acc[SETS];    // dU/dbeta of columns 4 b4 .. 4 b4 + 3, chain 4 s + j4
  double ul[SETS];    // likelihood part of U, chain 4 s + j4
#pragma unroll
  for (int s = 0; s < SETS; ++s) {
    acc[s] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    ul[s] = 0.0;
  }
  __syncthreads();  // beta
  for (int t = wa; t < ntiles; t += W) {
    const int rows = (int)min<int64_t>(TR, N - (int64_t)t * TR);
    if (t < full) {
#pragma unroll
      for (int j = 0; j < NLD; ++j)
        if (j < nld) *reinterpret_cast<f32x4*>(xs + dst[j]) = px[j];
      if (lane < TR) ys[wa][lane] = py;
      load(t + W);  // in flight during the compute below
    } else {  // the last rows, one number a lane; zeros after them
      const int64_t r0 = (int64_t)t * TR;
      const int ne = rows * D;
      for (int e = lane; e < TR * D; e += 64)
        xs[SD == D ? e : e + 4 * (e / D)] = e < ne ? X[r0 * D + e] : 0.0f;
      if (lane < TR) ys[wa][lane] = lane < rows ? Y[r0 + lane] : 0.0f;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    float yv[RV];
#pragma unroll
    for (int v = 0; v < RV; ++v) yv[v] = ys[wa][rl + v];
    // logits: lane = row (at TR = 32 twice), four interleaved sums
    const float* xr = xs + lane % TR * SD;
#pragma unroll
    for (int s0 = 0; s0 < SETS; s0 += SG) {
      f32x4 l[SG][4];
#pragma unroll
      for (int s = 0; s < SG; ++s)
#pragma unroll
        for (int k = 0; k < 4; ++k) l[s][k] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      if (quad) {
#pragma unroll 2
        for (int q = 0; q < D; q += 4) {
          const f32x4 xv = *reinterpret_cast<const f32x4*>(xr + q);
#pragma unroll
          for (int s = 0; s < SG; ++s) {
            const f32x4 bv = *reinterpret_cast<const f32x4*>(&beta[4 * (s0 + s) + j4][q]);
#pragma unroll
            for (int k = 0; k < 4; ++k)
              l[s][k] = __builtin_amdgcn_mfma_f32_4x4x1f32(xv[k], bv[k], l[s][k], 0, 0, 0);
          }
        }
      } else {
#pragma unroll 2
        for (int q = 0; q < D - 3; q += 4) {
#pragma unroll
          for (int s = 0; s < SG; ++s) {
            const f32x4 bv = *reinterpret_cast<const f32x4*>(&beta[4 * (s0 + s) + j4][q]);
#pragma unroll
            for (int k = 0; k < 4; ++k)
              l[s][k] = __builtin_amdgcn_mfma_f32_4x4x1f32(xr[q + k], bv[k], l[s][k], 0, 0, 0);
          }
        }
        const int q = D & ~3;
#pragma unroll
        for (int s = 0; s < SG; ++s) {
          const f32x4 bv = *reinterpret_cast<const f32x4*>(&beta[4 * (s0 + s) + j4][q]);
#pragma unroll
          for (int k = 0; k < 3; ++k)
            l[s][k] = __builtin_amdgcn_mfma_f32_4x4x1f32(q + k < D ? xr[q + k] : 0.0f, bv[k],
                                                         l[s][k], 0, 0, 0);
        }
      }
      // residuals, RV rows a lane from row rl; rows past `rows` get 0
#pragma unroll
      for (int s = 0; s < SG; ++s)
#pragma unroll
        for (int v = 0; v < RV; ++v) {
          f32x4 lv;
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            lv[k] = l[s][k][v];
            if (RV < 4 && upper) lv[k] = l[s][k][(v + RV) % 4];
          }
          float r, u;
          logistic_terms_f((lv[0] + lv[1]) + (lv[2] + lv[3]), yv[v], r, u);
          const bool ok = rl + v < rows;
          res[wa][4 * (s0 + s) + j4][rl + v] = ok ? r : 0.0f;
          ul[s0 + s] += ok ? (double)u : 0.0;
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // X^T R: lane = column, four interleaved sums over the tile's rows
    const float* xc = xs + lane;  // lanes past D: any number, not used
#pragma unroll
    for (int s0 = 0; s0 < SETS; s0 += SG) {
      f32x4 p[SG][4];
#pragma unroll
      for (int s = 0; s < SG; ++s)
#pragma unroll
        for (int k = 0; k < 4; ++k) p[s][k] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 2
      for (int n4 = 0; n4 < TR / 4; ++n4) {
#pragma unroll
        for (int s = 0; s < SG; ++s) {
          const f32x4 rv =
              *reinterpret_cast<const f32x4*>(&res[wa][4 * (s0 + s) + j4][4 * n4]);
#pragma unroll
          for (int k = 0; k < 4; ++k)
            p[s][k] = __builtin_amdgcn_mfma_f32_4x4x1f32(xc[(4 * n4 + k) * SD], rv[k],
                                                         p[s][k], 0, 0, 0);
        }
      }
#pragma unroll
      for (int s = 0; s < SG; ++s)
        acc[s0 + s] += (p[s][0] + p[s][1]) + (p[s][2] + p[s][3]);
    }
  }
#pragma unroll
  for (int s = 0; s < SETS; ++s) {
    *reinterpret_cast<f32x4*>(xs + (4 * s + j4) * kHierMaxD + 4 * b4) = acc[s];
#pragma unroll
    for (int o = 4; o < 64; o <<= 1) ul[s] += __shfl_xor(ul[s], o, 64);
    if (b4 == 0) rul[wa][4 * s + j4] = ul[s];
  }
  __syncthreads();
  for (int q = wa; q < K; q += W) {
    const int c = i * K + q;
    const float* z = zreq + (size_t)c * ldz;
    float* g = gout + (size_t)c * ldg;
    float a = 0.0f;
    double u = 0.0;
#pragma unroll
    for (int v = 0; v < W; ++v) {
      a += xs_all[v][q * kHierMaxD + lane];
      u += rul[v][q];
    }
    if (it.slot >= 0) {
      const size_t p = (size_t)it.slot * K + q;
      part_g[p * kHierMaxD + lane] = a;
      if (lane == 0) part_u[p] = u;
    } else {
      u = hier_finish(hd, D, lane, z, lane < D ? a : 0.0f, u, g);
      if (lane == 0) pe[c] = u;
    }
  }
}

// U and dU of the split models from their items' partial sums, added in row
// order: a wave per chain.
__global__ void __launch_bounds__(64)
hier_combine_kernel(HierData hd, const HierSplit* __restrict__ splits,
                    const float* __restrict__ part_g, const double* __restrict__ part_u,
                    const float* __restrict__ zreq, int ldz, double* __restrict__ pe,
                    float* __restrict__ gout, int ldg) {
  const HierSplit sp = splits[blockIdx.x / hd.K];
  const int q = blockIdx.x % hd.K, lane = threadIdx.x;
  const int D = hd.dims[sp.model];
  float a = 0.0f;
  double u = 0.0;
#pragma unroll 8
  for (int t = 0; t < sp.count; ++t) {
    const size_t p = (size_t)(sp.slot + t) * hd.K + q;
    a += part_g[p * kHierMaxD + lane];
    u += part_u[p];
  }
  const int c = sp.model * hd.K + q;
  u = hier_finish(hd, D, lane, zreq + (size_t)c * ldz, lane < D ? a : 0.0f, u,
                  gout + (size_t)c * ldg);
  if (lane == 0) pe[c] = u;
}

// One block per (model, chain subset): K chain slots of R waves each.  Wave
// r = 0 of a slot runs its chain's NUTS state machine; every wave of the
// block joins each gradient evaluation.
template <int K, int R, bool DENSE>
__global__ void __launch_bounds__(64 * K * R, (K * R <= 8) ? 2 : 1)
hier_persistent_kernel(HierData hd, EngineCfg cfg, Collect col,
                       const int64_t* __restrict__ d_target, ChainState* __restrict__ states,
                       float* __restrict__ vec, double* __restrict__ welf,
                       float* __restrict__ zreq, float* __restrict__ gout,
                       double* __restrict__ peout, int64_t* __restrict__ grad_evals) {
  __shared__ HierShared<K, R> sh;
  __shared__ int need_any;
  __shared__ ChainState sS[K];
  const int64_t target = *d_target;
  const int per = hd.K / K;  // workgroups per model
  const int i = hd.order[blockIdx.x / per];
  const int sub = blockIdx.x % per;
  const int wa = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int w = wa / R;
  const bool head = wa % R == 0;  // the wave that runs the state machine
  const int c = i * hd.K + sub * K + w;
  const ChainCtx cx = make_ctx<DENSE>(cfg, c, vec, welf);
  float* zr = zreq + (size_t)c * cfg.Dp;
  float* gi = gout + (size_t)c * cfg.Dp;
  ChainState& S = sS[w];
  if (head) copy_state(S, states[c], cx.lane);
  double pe = peout[c];
  int evals = 0;
  bool active = head;
  for (;;) {
    if (threadIdx.x == 0) need_any = 0;
    __syncthreads();
    bool need = false;
    if (active) {
      need = advance_chain(cfg, col, target, S, cx, c, zr, gi, pe, evals);
      active = need;
    }
    if (need && cx.lane == 0) atomicOr(&need_any, 1);
    __threadfence_block();
    __syncthreads();
    if (!need_any) break;
    const double u = hier_group_eval<K, R>(hd, i, sub, zreq, cfg.Dp, gout, cfg.Dp, sh);
    if (need) pe = u;
    __threadfence_block();
  }
  if (head) {
    copy_state(states[c], S, cx.lane);
    if (cx.lane == 0) {
      peout[c] = pe;
      if (evals && grad_evals) atomicAdd((unsigned long long*)grad_evals, (unsigned long long)evals);
    }
  }
}

__global__ void hier_chain_dims(const int* dims, int K, int C, int* out) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c < C) out[c] = dims[c / K] + 2;
}

struct HierPotential : Potential {
  HierData hd;
  int groups = 0, C = 0, maxd = 0;
  int* order = nullptr;
  int* dims = nullptr;
  int* cdims = nullptr;
  int64_t* row_off = nullptr;
  int64_t* elt_off = nullptr;
  double flops = 0.0, bytes = 0.0;
  // unforced evaluation: items heaviest first, the models of several items, and
  // the partial sums of those items
  HierItem* items = nullptr;
  HierSplit* splits = nullptr;
  float* part_g = nullptr;
  double* part_u = nullptr;
  int n_items = 0, n_splits = 0;
  // every model has at most 8 K rows: then a block's eight waves have hardly a tile
  // each and finish the chains one after the other, and a wave per chain on a
  // shared tile is faster (a call on 64 models, K = 16: 128 x 64 22.4 us against
  // 24.9, 256 x 64 28.1 against 27.1; K = 8: 8 x 64 17.4 against 22.6, 64 x 16 17.3
  // against 18.6, 128 x 64 19.9 against 19.5; K = 4: 8 x 64 17.4 against 21.0, 32 x 64
  // 17.5 against 18.1, 64 x 64 17.7 against 18.0)
  bool short_models = false;

  ~HierPotential() override {
    hipFree(items); hipFree(splits); hipFree(part_g); hipFree(part_u);
    hipFree(order); hipFree(dims); hipFree(cdims); hipFree(row_off); hipFree(elt_off);
  }
  int dim() const override { return maxd + 2; }
  const char* name() const override { return "hier"; }
  bool set_positive_transform(int kind) override {
    hd.softplus = kind == 1;
    return true;
  }
  bool persistent() const override { return true; }
  const int* chain_dims() const override { return cdims; }
  double alg_bytes(int) const override { return bytes; }
  double alg_flops(int) const override { return flops; }

  // launch shape: kb chains per workgroup (a divisor of hd.K; 0: hd.K) and
  // rw waves per chain, code = kb + 32 (rw - 1).  The default (hd.K, 1) runs
  // until iteration kHierTuneAt, where the tuned shape (kb_t, rw_t) takes
  // over -- timed on trees of working size, not the first iterations' few
  // leaves -- unless a shape was fixed.
  static constexpr int64_t kHierTuneAt = 50;
  int kb = 0, rw = 1;
  int kb_t = 0, rw_t = 1;
  std::string tuned_log;
  int tuned_chains = 0;
  bool forced = false;
  HierPotential() { tune_at = kHierTuneAt; }
  static int shape_code(int k, int r) { return k + 32 * (r - 1); }
  static std::string shape_label(int code) {
    return std::to_string(code % 32) + "x" + std::to_string(code / 32 + 1);
  }
  // the (kb, rw) pairs with a kernel: rw in {1, 2, 4}, kb rw <= 16
  static bool has_kernel(int k, int r) {
    return (r == 1 && (k == 1 || k == 2 || k == 4 || k == 8 || k == 16)) ||
           ((r == 2 || r == 4) && (k == 1 || k == 2 || k == 4) && k * r <= 16);
  }
  void describe(const std::string& how) {
    tuning = "hier: " + std::to_string(waves()) + " chains per workgroup of " +
             std::to_string(hd.K) + " per model, " + std::to_string(rw) +
             " waves per chain " + how;
  }
  bool force_launch_shape(int shape) override {
    const int k = shape % 32, r = shape / 32 + 1;
    if (k < 1 || k > hd.K || hd.K % k || !has_kernel(k, r)) return false;
    kb = k;
    rw = r;
    forced = true;
    tune_at = 0;
    describe("(fixed)");
    return true;
  }

  int waves() const { return kb > 0 ? kb : hd.K; }

  hipError_t eval(hipStream_t s, const float* z, int ldz, int Cn, double* pe, float* g,
                  int ldg) override {
    if (Cn != C || ldz < maxd + 2 || ldg < maxd + 2) return hipErrorInvalidValue;
    // one evaluation of every chain, unless a shape was fixed: then that shape's
    // evaluation, whose sums are in the order of the persistent launch's
    bool launched = false;
    mark_begin(s);
    if (!forced && !short_models) {
#define NAX_K(KV)                                                                             \
  if (hd.K == KV)                                                                             \
    hipLaunchKernelGGL((hier_once_kernel<KV, kOnceWaves, kOnceRows>), dim3(n_items),          \
                       dim3(64 * kOnceWaves), 0, s, hd, items, z, ldz, pe, g, ldg, part_g,    \
                       part_u);
      NAX_K(1) NAX_K(2) NAX_K(4) NAX_K(8) NAX_K(16)
#undef NAX_K
      if (n_splits)
        hipLaunchKernelGGL(hier_combine_kernel, dim3(n_splits * hd.K), dim3(64), 0, s, hd, splits,
                           part_g, part_u, z, ldz, pe, g, ldg);
      mark_end(s);
      return hipGetLastError();
    }
    const int w = waves(), r = forced ? rw : 1;
    const dim3 grid(groups * (hd.K / w));
#define NAX_KR(KV, RV)                                                                        \
  if (!launched && w == KV && r == RV) {                                                      \
    hipLaunchKernelGGL((hier_eval_kernel<KV, RV>), grid, dim3(64 * KV * RV), 0, s, hd, z,     \
                       ldz, pe, g, ldg);                                                      \
    launched = true;                                                                          \
  }
    NAX_KR(1, 1) NAX_KR(2, 1) NAX_KR(4, 1) NAX_KR(8, 1) NAX_KR(16, 1)
    NAX_KR(1, 2) NAX_KR(2, 2) NAX_KR(4, 2)
    NAX_KR(1, 4) NAX_KR(2, 4) NAX_KR(4, 4)
#undef NAX_KR
    if (!launched) return hipErrorInvalidValue;
    mark_end(s);
    return hipGetLastError();
  }

  hipError_t launch(int code, hipStream_t s, const EngineCfg& cfg, const Collect& col,
                    const int64_t* d_target, ChainState* st, float* vec, double* wel, float* zreq,
                    float* gout, double* peout, int64_t* gevals) const {
    const int w = code % 32, r = code / 32 + 1;
    if (w < 1 || hd.K % w) return hipErrorInvalidValue;
    const dim3 grid(groups * (hd.K / w));
#define NAX_KR(KV, RV)                                                                        \
  if (w == KV && r == RV) {                                                                   \
    if (cfg.dense)                                                                            \
      hipLaunchKernelGGL((hier_persistent_kernel<KV, RV, true>), grid, dim3(64 * KV * RV), 0,  \
                         s, hd, cfg, col, d_target, st, vec, wel, zreq, gout, peout, gevals); \
    else                                                                                      \
      hipLaunchKernelGGL((hier_persistent_kernel<KV, RV, false>), grid, dim3(64 * KV * RV), 0, \
                         s, hd, cfg, col, d_target, st, vec, wel, zreq, gout, peout, gevals); \
    return hipGetLastError();                                                                 \
  }
    NAX_KR(1, 1) NAX_KR(2, 1) NAX_KR(4, 1) NAX_KR(8, 1) NAX_KR(16, 1)
    NAX_KR(1, 2) NAX_KR(2, 2) NAX_KR(4, 2)
    NAX_KR(1, 4) NAX_KR(2, 4) NAX_KR(4, 4)
#undef NAX_KR
    return hipErrorInvalidValue;
  }

  hipError_t prepare_persistent(hipStream_t s, const EngineCfg& cfg, ChainState* st, float* vec,
                                double* wel, float* zreq, float* gout, double* peout) override {
    // candidates: one workgroup per model (kb = K) with 1, 2 or 4 waves per
    // chain, or each model's chains split over 2 or 4 workgroups (K/2, K/4)
    // with one wave each; timed over 5 iterations from a scratch copy of
    // the state.  The choice is kept per process for this shape of workload
    // (the waves per chain set the order of the sums, so the draws).
    if (forced) return hipSuccess;
    if (chain_iter < tune_at) {
      kb = 0;
      rw = 1;
      describe("(default until iteration " + std::to_string(tune_at) + ", then tuned)");
      return hipSuccess;
    }
    if (kb_t == 0 || tuned_chains != cfg.C) {
      const std::string key = "hier G=" + std::to_string(groups) + " K=" + std::to_string(hd.K) +
                              " C=" + std::to_string(cfg.C) + " dense=" + std::to_string(cfg.dense);
      int code = 0;
      if (tuned_shape(key, &code, false)) {
        tuned_log = "(tuned earlier in this process)";
      } else {
        std::vector<int> cands;
        for (int r : {1, 2, 4})
          if (has_kernel(hd.K, r)) cands.push_back(shape_code(hd.K, r));
        for (int w = hd.K / 2; w >= 1 && w * 4 >= hd.K; w /= 2)
          if (has_kernel(w, 1)) cands.push_back(shape_code(w, 1));
        std::string log;
        auto go = [&](int c, hipStream_t ss, const Collect& col, const int64_t* tgt,
                      ChainState* st2, float* vec2, double* wel2, float* zr2, float* g2,
                      double* pe2, int64_t* ge2) {
          return launch(c, ss, cfg, col, tgt, st2, vec2, wel2, zr2, g2, pe2, ge2);
        };
        code = tune_persistent(s, cfg, st, vec, wel, zreq, gout, peout, 5, cands, go, &log,
                               &HierPotential::shape_label);
        tuned_shape(key, &code, true);
        tuned_log = "(from iteration " + std::to_string(tune_at) +
                    "; ms for 5 iterations, chains per workgroup x waves per chain:" + log + ")";
      }
      kb_t = code % 32;
      rw_t = code / 32 + 1;
      tuned_chains = cfg.C;
    }
    kb = kb_t;
    rw = rw_t;
    describe(tuned_log);
    return hipSuccess;
  }

  hipError_t run_persistent(hipStream_t s, const EngineCfg& cfg, const Collect& col,
                            const int64_t* d_target, ChainState* st, float* vec, double* wel,
                            float* zreq, float* gout, double* peout, int64_t* gevals) override {
    mark_begin(s);
    const hipError_t e = launch(shape_code(waves(), rw), s, cfg, col, d_target, st, vec, wel,
                                zreq, gout, peout, gevals);
    mark_end(s);
    return e;
  }
};

Potential* make_hier(const float* x, const float* y, const int64_t* d_row_off,
                     const int64_t* d_elt_off, const int* d_dims, int groups, int K, int C,
                     int Dp, hipStream_t s, std::string* err) {
  if (K != 1 && K != 2 && K != 4 && K != 8 && K != 16) {
    *err = "hierarchical model: chains_per_group must be 1, 2, 4, 8 or 16";
    return nullptr;
  }
  std::vector<int> hd_dims(groups);
  std::vector<int64_t> hrow(groups + 1), helt(groups);
  if (hipMemcpy(hd_dims.data(), d_dims, sizeof(int) * groups, hipMemcpyDeviceToHost) != hipSuccess ||
      hipMemcpy(hrow.data(), d_row_off, sizeof(int64_t) * (groups + 1), hipMemcpyDeviceToHost) != hipSuccess ||
      hipMemcpy(helt.data(), d_elt_off, sizeof(int64_t) * groups, hipMemcpyDeviceToHost) != hipSuccess) {
    *err = "hierarchical model: cannot read the group tables";
    return nullptr;
  }
  auto* p = new HierPotential();
  p->groups = groups;
  p->C = C;
  double work = 0.0;
  int64_t longest = 0;
  std::vector<double> w(groups);
  for (int i = 0; i < groups; ++i) {
    const int64_t n = hrow[i + 1] - hrow[i];
    if (hd_dims[i] < 1 || hd_dims[i] > kHierMaxD || n < 1) {
      *err = "hierarchical model: every group needs 1 <= D_i <= 64 and N_i >= 1";
      delete p;
      return nullptr;
    }
    p->maxd = std::max(p->maxd, hd_dims[i]);
    longest = std::max(longest, n);
    w[i] = (double)n * hd_dims[i];
    work += w[i];
  }
  p->short_models = longest <= 8 * K;
  p->flops = 4.0 * K * work;         // x.beta and X^T r per chain
  p->bytes = 4.0 * work + 4.0 * (double)(hrow[groups] - hrow[0]);  // X once per model + labels
  std::vector<int> ord(groups);
  std::iota(ord.begin(), ord.end(), 0);
  std::stable_sort(ord.begin(), ord.end(), [&](int a, int b) { return w[a] > w[b]; });
  std::vector<HierItem> items;
  std::vector<HierSplit> splits;
  const double share = std::max(work / kOnceItems, kOnceItemMin);
  int slots = 0;
  for (int i : ord) {
    const int64_t n = hrow[i + 1] - hrow[i];
    const int64_t tiles = (n + kOnceRows - 1) / kOnceRows;
    const int64_t parts = std::min<int64_t>(tiles, (int64_t)std::ceil(w[i] / share));
    if (parts > 1) splits.push_back({i, slots, (int)parts});
    for (int64_t t = 0; t < parts; ++t) {
      const int64_t a = tiles * t / parts * kOnceRows;
      const int64_t b = std::min<int64_t>(n, tiles * (t + 1) / parts * kOnceRows);
      items.push_back({a, b - a, i, parts > 1 ? slots++ : -1});
    }
  }
  std::stable_sort(items.begin(), items.end(), [&](const HierItem& a, const HierItem& b) {
    return a.rows * hd_dims[a.model] > b.rows * hd_dims[b.model];
  });
  p->n_items = (int)items.size();
  p->n_splits = (int)splits.size();
  hipError_t e = hipMalloc(&p->order, sizeof(int) * groups);
  if (e == hipSuccess) e = hipMalloc(&p->items, sizeof(HierItem) * items.size());
  if (e == hipSuccess && slots) {
    e = hipMalloc(&p->splits, sizeof(HierSplit) * splits.size());
    if (e == hipSuccess) e = hipMalloc(&p->part_g, sizeof(float) * slots * K * kHierMaxD);
    if (e == hipSuccess) e = hipMalloc(&p->part_u, sizeof(double) * slots * K);
    if (e == hipSuccess) e = hipMemcpy(p->splits, splits.data(), sizeof(HierSplit) * splits.size(), hipMemcpyHostToDevice);
  }
  if (e == hipSuccess) e = hipMemcpy(p->items, items.data(), sizeof(HierItem) * items.size(), hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMalloc(&p->dims, sizeof(int) * groups);
  if (e == hipSuccess) e = hipMalloc(&p->cdims, sizeof(int) * C);
  if (e == hipSuccess) e = hipMalloc(&p->row_off, sizeof(int64_t) * (groups + 1));
  if (e == hipSuccess) e = hipMalloc(&p->elt_off, sizeof(int64_t) * groups);
  if (e == hipSuccess) e = hipMemcpy(p->order, ord.data(), sizeof(int) * groups, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(p->dims, hd_dims.data(), sizeof(int) * groups, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(p->row_off, hrow.data(), sizeof(int64_t) * (groups + 1), hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(p->elt_off, helt.data(), sizeof(int64_t) * groups, hipMemcpyHostToDevice);
  if (e != hipSuccess) {
    *err = std::string("hierarchical model: ") + hipGetErrorString(e);
    delete p;
    return nullptr;
  }
  hipLaunchKernelGGL(hier_chain_dims, dim3((C + 255) / 256), dim3(256), 0, s, p->dims, K, C, p->cdims);
  e = hipStreamSynchronize(s);
  if (e != hipSuccess) {
    *err = std::string("hierarchical model: ") + hipGetErrorString(e);
    delete p;
    return nullptr;
  }
  p->hd = HierData{x, y, p->row_off, p->elt_off, p->dims, p->order, K, Dp, 0};
  return p;
}

}  // namespace nax
