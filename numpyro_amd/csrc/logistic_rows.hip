// The logistic potential for a few chains of a fp32 design: U and dU of up to 16
// chains per workgroup from wave-owned tiles of 32 rows.
//
// A call reads X once for 16 chains, so with few chains it is bound by that read,
// and the work per element has to stay far below it.  Each wave owns its tiles (no
// barrier in the loop): 16 bytes a lane loaded into registers one tile ahead,
// stored to the wave's LDS tile, then
//   logits     lane = row: one v_mfma_f32_4x4x1 (16 blocks of 4 rows x 4 chains) per
//              column and 4 chains, the fused multiply-adds over the columns in order,
//              bit for bit those of logit_partial_f32
//   residuals  lane = (2 rows, chain)
//   X^T R      lane = column: one v_mfma_f32_4x4x1 per row, 64 columns and 4 chains
// The block's waves are added in wave order into its row-split partial, and
// logit_reduce adds the partials and the prior.
// Bound: the read of X up to about 8 chains (581,012 x 55, 1 chain, 130 MB: the tile
// kernel, one chain of its eight in use and three barriers a tile, 81 us; 38 us now,
// 3.4 TB/s; 1,000,000 x 256, 1 chain, 1.02 GB: 0.29 ms a pass); the 4x4x1 products past
// that, where at 256 columns the LDS leaves one wave per SIMD to hide their latency.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <string>

#include "nax_device.h"
#include "nax_internal.h"

namespace nax {
namespace {

constexpr int kRowsWaves = 4;  // waves of a block
constexpr int kRowsTile = 32;  // rows of a wave's tile
constexpr int kRowsMaxD = 256;
// fourth word of a buffer descriptor: plain 32-bit data
constexpr int kBufferWord3 = 0x00027000;

typedef float f32x4 __attribute__((ext_vector_type(4)));

// CB = ceil(D / 64) column blocks, SETS groups of 4 chains.
template <int CB, int SETS>
struct RowsShared {
  static constexpr int LD = 64 * CB + 4;
  // each wave's X tile, at the end its partial X^T R ([chain][column])
  __attribute__((aligned(16))) float xs[kRowsWaves][kRowsTile * LD];
  __attribute__((aligned(16))) float beta[4 * SETS][LD];  // chains past C: 0
  __attribute__((aligned(16))) float res[kRowsWaves][4 * SETS][kRowsTile + 4];
  __attribute__((aligned(16))) float ys[kRowsWaves][kRowsTile];
  double rul[kRowsWaves][4 * SETS];
};

template <int CB, int SETS>
__global__ void __launch_bounds__(64 * kRowsWaves, CB > 2 ? 1 : 2)
logit_rows_kernel(const float* __restrict__ X, const float* __restrict__ Y, int64_t N, int D,
                  const float* __restrict__ Z, int ldz, int C, float* __restrict__ wsg,
                  double* __restrict__ wsu) {
  constexpr int W = kRowsWaves, TR = kRowsTile, NC = 4 * SETS;
  constexpr int NLD = TR * 64 * CB / 256;  // 16-byte loads of a tile
  __shared__ RowsShared<CB, SETS> sh;
  const int wa = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int lane = threadIdx.x & 63;
  const int c0 = blockIdx.y * NC;
  const int64_t nt = (N + TR - 1) / TR, full = N / TR;
  const int64_t step = (int64_t)gridDim.x * W;
  float* xs = sh.xs[wa];
  // Rows are SD apart in LDS: D a multiple of 8 takes 4 floats of padding, which
  // spreads the rows over the banks; any other D is conflict-free (or 2-way).
  const bool quad = (D & 3) == 0;
  const int SD = (D & 7) == 0 ? D + 4 : D;
  const int nld = (TR * D + 255) / 256;
  int dst[NLD];
#pragma unroll
  for (int j = 0; j < NLD; ++j) {
    const int e = 4 * (lane + 64 * j);
    dst[j] = SD == D ? e : e + 4 * (e / D);
  }
  f32x4 px[NLD];
  float py = 0.0f;
  // Every load of a full tile is issued, without a branch: what lies past the
  // tile's TR D elements (16 bytes never straddle that end) or past the last full
  // tile reads as 0 and takes no memory access.
  auto load = [&](int64_t t) {
    const int64_t r0 = t * TR;
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
  const int64_t t0 = (int64_t)wa * gridDim.x + blockIdx.x;
  load(t0);
  for (int q = wa; q < NC; q += W)
#pragma unroll
    for (int b = 0; b < CB; ++b) {
      const int d = 64 * b + lane;
      sh.beta[q][d] = c0 + q < C && d < D ? Z[(size_t)(c0 + q) * ldz + d] : 0.0f;
    }
  const int j4 = lane & 3, b4 = lane >> 2;  // chain of a set, block of 4 rows / columns
  // Blocks 8..15 repeat the rows of blocks 0..7; a lane takes the residuals of the
  // first or last two of its block's four rows.
  const bool upper = lane >= TR;
  const int rl = 4 * b4 % TR + (upper ? 2 : 0);
  f32x4 acc[CB][SETS];  // dU/dbeta of columns 64 b + 4 b4 .. + 3, chain 4 s + j4
  CompSum ul[SETS];     // likelihood part of U, chain 4 s + j4
#pragma unroll
  for (int b = 0; b < CB; ++b)
#pragma unroll
    for (int s = 0; s < SETS; ++s) acc[b][s] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  __syncthreads();  // beta
  for (int64_t t = t0; t < nt; t += step) {
    const int rows = (int)min<int64_t>(TR, N - t * TR);
    if (t < full) {
#pragma unroll
      for (int j = 0; j < NLD; ++j)
        if (j < nld) *reinterpret_cast<f32x4*>(xs + dst[j]) = px[j];
      if (lane < TR) sh.ys[wa][lane] = py;
      load(t + step);  // in flight during the compute below
    } else {  // the last rows, one number a lane; zeros after them
      const int64_t r0 = t * TR;
      const int ne = rows * D;
      for (int e = lane; e < TR * D; e += 64)
        xs[SD == D ? e : e + 4 * (e / D)] = e < ne ? X[r0 * D + e] : 0.0f;
      if (lane < TR) sh.ys[wa][lane] = lane < rows ? Y[r0 + lane] : 0.0f;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const float* xr = xs + lane % TR * SD;
    const float* br = &sh.beta[j4][0];
    constexpr int LB = 4 * RowsShared<CB, SETS>::LD;  // to the next set's chain
    f32x4 l[SETS];
#pragma unroll
    for (int s = 0; s < SETS; ++s) l[s] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    if (quad) {
#pragma unroll 2
      for (int q = 0; q < D; q += 4) {
        const f32x4 xv = *reinterpret_cast<const f32x4*>(xr + q);
#pragma unroll
        for (int s = 0; s < SETS; ++s) {
          const f32x4 bv = *reinterpret_cast<const f32x4*>(br + s * LB + q);
#pragma unroll
          for (int k = 0; k < 4; ++k)
            l[s] = __builtin_amdgcn_mfma_f32_4x4x1f32(xv[k], bv[k], l[s], 0, 0, 0);
        }
      }
    } else {
#pragma unroll 2
      for (int q = 0; q < D - 3; q += 4) {
#pragma unroll
        for (int s = 0; s < SETS; ++s) {
          const f32x4 bv = *reinterpret_cast<const f32x4*>(br + s * LB + q);
#pragma unroll
          for (int k = 0; k < 4; ++k)
            l[s] = __builtin_amdgcn_mfma_f32_4x4x1f32(xr[q + k], bv[k], l[s], 0, 0, 0);
        }
      }
      for (int q = D & ~3; q < D; ++q)
#pragma unroll
        for (int s = 0; s < SETS; ++s)
          l[s] = __builtin_amdgcn_mfma_f32_4x4x1f32(xr[q], br[s * LB + q], l[s], 0, 0, 0);
    }
    const float y0 = sh.ys[wa][rl], y1 = sh.ys[wa][rl + 1];
#pragma unroll
    for (int s = 0; s < SETS; ++s)
#pragma unroll
      for (int v = 0; v < 2; ++v) {
        const float lv = upper ? l[s][v + 2] : l[s][v], yv = v ? y1 : y0;
        const bool ok = rl + v < rows;
        sh.res[wa][4 * s + j4][rl + v] = ok ? sigmoidf_(lv) - yv : 0.0f;
        if (ok) ul[s].add((double)(softplusf_(lv) - yv * lv));
      }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const float* xc = xs + lane;  // columns past D: any number, not used
#pragma unroll
    for (int b = 0; b < CB; ++b) {
      f32x4 p[SETS][2];  // even and odd rows of the tile
#pragma unroll
      for (int s = 0; s < SETS; ++s) p[s][0] = p[s][1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 2
      for (int n4 = 0; n4 < TR / 4; ++n4) {
        float xv[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) xv[k] = xc[(4 * n4 + k) * SD + 64 * b];
#pragma unroll
        for (int s = 0; s < SETS; ++s) {
          const f32x4 rv = *reinterpret_cast<const f32x4*>(&sh.res[wa][4 * s + j4][4 * n4]);
#pragma unroll
          for (int k = 0; k < 4; ++k)
            p[s][k & 1] = __builtin_amdgcn_mfma_f32_4x4x1f32(xv[k], rv[k], p[s][k & 1], 0, 0, 0);
        }
      }
#pragma unroll
      for (int s = 0; s < SETS; ++s) acc[b][s] += p[s][0] + p[s][1];
    }
  }
#pragma unroll
  for (int s = 0; s < SETS; ++s) {
#pragma unroll
    for (int b = 0; b < CB; ++b)
      *reinterpret_cast<f32x4*>(xs + (4 * s + j4) * 64 * CB + 64 * b + 4 * b4) = acc[b][s];
#pragma unroll
    for (int o = 4; o < 64; o <<= 1) {
      CompSum v;
      v.s = __shfl_xor(ul[s].s, o, 64);
      v.c = __shfl_xor(ul[s].c, o, 64);
      ul[s].add(v);
    }
    if (b4 == 0) sh.rul[wa][4 * s + j4] = ul[s].value();
  }
  __syncthreads();
  const int nc = min(NC, C - c0);
  for (int e = threadIdx.x; e < nc * 64 * CB; e += 64 * W) {
    const int q = e / (64 * CB), d = e % (64 * CB);
    if (d < D) {
      float a = 0.0f;
#pragma unroll
      for (int v = 0; v < W; ++v) a += sh.xs[v][e];
      wsg[((size_t)blockIdx.x * C + c0 + q) * D + d] = a;
    }
  }
  if ((int)threadIdx.x < nc) {
    CompSum u;
#pragma unroll
    for (int v = 0; v < W; ++v) u.add(sh.rul[v][threadIdx.x]);
    wsu[(size_t)blockIdx.x * C + c0 + threadIdx.x] = u.value();
  }
}

struct RowsPotential : Potential {
  const float* x = nullptr;
  const float* y = nullptr;
  int64_t n = 0;
  int d = 0;
  double prior_scale = 1.0;
  float* wsg = nullptr;
  double* wsu = nullptr;
  size_t slots = 0;  // row splits x chains the workspaces hold

  ~RowsPotential() override {
    hipFree(wsg);
    hipFree(wsu);
  }
  int dim() const override { return d; }
  const char* name() const override { return "logit_rows_f32"; }
  double alg_bytes(int C) const override { return 4.0 * (double)n * d + 4.0 * n; }
  double alg_flops(int C) const override { return 4.0 * (double)n * d * C; }

  // Row splits of C chains: as many blocks as the chip's LDS holds, divided by the
  // chain tiles, and evened out so that every wave has the same number of tiles.
  int row_splits(size_t lds, int chain_tiles) const {
    const int64_t fit =
        std::max<int64_t>(1, 256 * std::min<int64_t>(4, (160 << 10) / lds) / chain_tiles);
    const int64_t nt = (n + kRowsTile - 1) / kRowsTile;
    const int64_t per = (nt + fit * kRowsWaves - 1) / (fit * kRowsWaves);
    return (int)((nt + per * kRowsWaves - 1) / (per * kRowsWaves));
  }

  template <int CB, int SETS>
  hipError_t run(hipStream_t s, const float* z, int ldz, int C, double* pe, float* g, int ldg) {
    const int ct = (C + 4 * SETS - 1) / (4 * SETS);
    const int RB = row_splits(sizeof(RowsShared<CB, SETS>), ct);
    if (slots < (size_t)RB * C) {
      hipFree(wsg);
      hipFree(wsu);
      wsg = nullptr;
      wsu = nullptr;
      slots = 0;
      hipError_t e = hipMalloc(&wsg, sizeof(float) * (size_t)RB * C * d);
      if (e == hipSuccess) e = hipMalloc(&wsu, sizeof(double) * (size_t)RB * C);
      if (e != hipSuccess) return e;
      slots = (size_t)RB * C;
    }
    mark_begin(s);
    hipLaunchKernelGGL((logit_rows_kernel<CB, SETS>), dim3(RB, ct), dim3(64 * kRowsWaves), 0, s, x,
                       y, n, d, z, ldz, C, wsg, wsu);
    mark_end(s);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const double inv_s2 = 1.0 / (prior_scale * prior_scale);
    const double log_norm = std::log(std::sqrt(2.0 * M_PI) * prior_scale);
    hipLaunchKernelGGL(logit_reduce, dim3(C), dim3(reduce_threads(C)), 0, s, wsg, wsu, RB, C, d, z,
                       ldz, inv_s2, log_norm, 0.0, pe, g, ldg, nullptr, nullptr, 0, 0);
    return hipGetLastError();
  }

  hipError_t eval(hipStream_t s, const float* z, int ldz, int C, double* pe, float* g,
                  int ldg) override {
    const int cb = (d + 63) / 64, sets = C <= 4 ? 1 : C <= 8 ? 2 : 4;
#define NAX_ROWS(CB, SETS) \
  if (cb == CB && sets == SETS) return run<CB, SETS>(s, z, ldz, C, pe, g, ldg);
    NAX_ROWS(1, 1) NAX_ROWS(1, 2) NAX_ROWS(1, 4) NAX_ROWS(2, 1) NAX_ROWS(2, 2) NAX_ROWS(2, 4)
    NAX_ROWS(3, 1) NAX_ROWS(3, 2) NAX_ROWS(3, 4) NAX_ROWS(4, 1) NAX_ROWS(4, 2) NAX_ROWS(4, 4)
#undef NAX_ROWS
    return hipErrorInvalidValue;
  }
};

}  // namespace

Potential* make_logistic_rows(const float* x, const float* y, int64_t n, int d,
                              double prior_scale) {
  if (d > kRowsMaxD) return nullptr;
  auto* p = new RowsPotential();
  p->x = x;
  p->y = y;
  p->n = n;
  p->d = d;
  p->prior_scale = prior_scale;
  return p;
}

}  // namespace nax
