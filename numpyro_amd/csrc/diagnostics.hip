// On-device MCMC diagnostics over collected draws x [C chains][S draws][P]
// (the layout nax_run collects z in): effective sample size with Geyer's
// initial monotone sequence and split Gelman-Rubin, per parameter
// (numpyro/diagnostics.py:158-203, 64-80, 29-42).  The reference computes the
// autocovariance by FFT; here the (biased) autocovariances
// sum_t xc_t xc_{t+k} / S are lag products summed in fp64.
//
// Two facts set the shape of the work.  The parameters are the fastest index
// of x, so a workgroup takes a tile of PT neighbouring parameters (lanes along
// them: a row of the tile is one coalesced read) of one chain at a time, for
// a group of chains.  And the initial monotone sequence is clipped at zero:
// from the first pair of lags whose sum is not positive on, every later pair
// adds nothing.  So lags are computed 32 at a time for all chains
// (diag_lags_kernel), diag_finish_kernel advances each parameter's sequence
// over them, and only tiles with a parameter whose sequence is still positive
// get more lags.
//
// Bound: fp64 multiply-adds of the lag products (16 per draw read and pass),
// then the read of x.  128 chains x 600 draws x 3002 parameters: 37.4 ms with
// a workgroup per parameter that computed all S lags from strided reads (each
// 4-byte read of x fetched a whole cache line), 1.76 ms with these kernels
// (0.64 ms of it the first 32 lags of every parameter).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>

#include "nax_device.h"
#include "nax_internal.h"

namespace nax {

constexpr int kDiagMaxDraws = 4096;
constexpr int kDiagThreads = 512;
constexpr int kDiagLpt = 16;      // lags per thread: a sliding window of registers
constexpr int kDiagGroups = 2;    // lag groups of a pass
constexpr int kDiagPass = kDiagLpt * kDiagGroups;  // 32 lags per pass

// Welford over chains of (mean, variance) pairs.
struct ChainAgg {
  int n = 0;
  double mean_of_means = 0.0, m2_of_means = 0.0, sum_var = 0.0;
  __device__ void add(double m, double v) {
    n += 1;
    const double d = m - mean_of_means;
    mean_of_means += d / n;
    m2_of_means += d * (m - mean_of_means);
    sum_var += v;
  }
  // the chains of another aggregate (parallel form of the same update)
  __device__ void merge(int on, double omean, double om2, double osum) {
    if (on == 0) return;
    const double d = omean - mean_of_means;
    const int t = n + on;
    mean_of_means += d * on / t;
    m2_of_means += om2 + d * d * ((double)n * on / t);
    sum_var += osum;
    n = t;
  }
  // _compute_chain_variance_stats: (var_within, var_estimator) for chains of
  // length len
  __device__ void stats(int len, double& vw, double& ve) const {
    vw = sum_var / n;
    ve = vw * (len - 1) / len;
    if (n > 1) ve += m2_of_means / (n - 1);
    else vw = ve;
  }
};

// Chains [diag_chain(g), diag_chain(g + 1)) belong to chain group g of ng.
__host__ __device__ inline int diag_chain(int C, int g, int ng) {
  return (int)((int64_t)C * g / ng);
}

constexpr int kAggDoubles = 6;  // full and split (mean of means, m2 of means, sum of variances)

// Sums of NV values over the threads of a column (tid % PT), for every thread:
// inside the wave by shuffles, then the waves' partials in wave order.
template <int PT, int NV>
__device__ __forceinline__ void column_sums(double (&v)[NV], double* red) {
  const int lane = threadIdx.x & (NAX_WAVE - 1), wave = threadIdx.x / NAX_WAVE;
  constexpr int NW = kDiagThreads / NAX_WAVE;
#pragma unroll
  for (int i = 0; i < NV; ++i)
#pragma unroll
    for (int o = NAX_WAVE / 2; o >= PT; o >>= 1) v[i] += __shfl_xor(v[i], o, NAX_WAVE);
  __syncthreads();  // earlier readers of red are done
  if (lane < PT)
#pragma unroll
    for (int i = 0; i < NV; ++i) red[(i * NW + wave) * PT + lane] = v[i];
  __syncthreads();
  const int p = threadIdx.x % PT;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    double t = 0.0;
#pragma unroll
    for (int w = 0; w < NW; ++w) t += red[(i * NW + w) * PT + p];
    v[i] = t;
  }
}

// One workgroup: tile of PT parameters, the chains of one group, 32 lags from
// base + 32 blockIdx.y on.  Threads: p = tid % PT, lag group (16 lags) and
// time segment.  A chain's tile sits in LDS as fp32; each thread slides a
// window of 16 centred values along its segment, so one new value and one
// multiplicand are read and converted per 16 multiply-adds (first pass of
// 128 x 600 x 3002: 1.11 ms at 8 lags per thread, 0.98 at 16, 0.64 with the tile
// loaded straight to LDS).  The sums run on over the
// group's chains and are combined over the segments once, at the end.
// blockIdx.x maps to (tile, group) such that an XCD's workgroups take
// neighbouring tiles of the same chains (rows that share cache lines).
// tiles: the nt tiles to do, or null for all; agg: written by the first pass.
// x holds P parameters at a row stride of ldx.
template <int PT>
__global__ void __launch_bounds__(kDiagThreads, 4)
diag_lags_kernel(const float* __restrict__ x, int C, int S, int P, int ldx,
                 const int* __restrict__ tiles, int nt, int ng, int base, double* __restrict__ gpart, double* __restrict__ agg) {
  constexpr int NSUB = kDiagThreads / PT;
  constexpr int NSEG = NSUB / kDiagGroups;
  extern __shared__ __attribute__((aligned(16))) float xs[];  // [S][PT]; then the segment sums
  __shared__ double red[2 * (kDiagThreads / NAX_WAVE) * PT];
  const int per = (nt * ng + 7) / 8;
  const int id = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || id >= nt * ng) return;
  const int g = id / nt, pos = id % nt;
  const int tile = tiles ? tiles[pos] : pos;
  const int tid = threadIdx.x;
  const int p = tid % PT, sub = tid / PT;
  const int grp = sub % kDiagGroups, seg = sub / kDiagGroups;
  const int p0 = tile * PT;
  const bool pvalid = p0 + p < P;
  const int k0 = base + kDiagPass * (int)blockIdx.y + kDiagLpt * grp;
  const int klast = base + kDiagPass * (int)blockIdx.y + kDiagPass - 1;  // of the whole pass
  const int len = ((S + NSEG - 1) / NSEG + kDiagLpt - 1) / kDiagLpt * kDiagLpt;
  const int t0 = seg * len;
  const int t1 = min(S - k0, min(S, t0 + len));  // products of lag k0 end at S - k0
  const bool stats = agg != nullptr && blockIdx.y == 0;
  const int h = S / 2;
  double acc[kDiagLpt];
#pragma unroll
  for (int j = 0; j < kDiagLpt; ++j) acc[j] = 0.0;
  ChainAgg ag;  // of the whole chains on even threads of a column, of the halves on odd ones
  const int c1 = diag_chain(C, g + 1, ng);
  for (int c = diag_chain(C, g, ng); c < c1; ++c) {
    __syncthreads();  // the previous chain's tile is no longer read
    const float* xc = x + (size_t)c * S * ldx + p0 + p;
    // straight to LDS: every load of the tile is in flight at once, in no
    // register.  A wave's 64 lanes are 64 / PT consecutive rows of the tile;
    // columns past P are not read (and nothing of them is written).
    for (int t = sub; t < S; t += NSUB)
      if (pvalid)
        lds_dma4(xc + (size_t)t * ldx,
                 lds_addr(xs + __builtin_amdgcn_readfirstlane(t) * PT));
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    // sums of the halves [0, h) and [S - h, S); S odd leaves the middle draw
    double m[2] = {0.0, 0.0};
    for (int t = sub; t < h; t += NSUB) {
      m[0] += (double)xs[t * PT + p];
      m[1] += (double)xs[(S - h + t) * PT + p];
    }
    column_sums<PT, 2>(m, red);
    const double mid = (S & 1) ? (double)xs[h * PT + p] : 0.0;
    const double mean = (m[0] + m[1] + mid) / S;
    if (stats) {
      // the halves centred on their own means, and the whole chain's squares
      // from theirs (a sum of squares each: nothing cancels)
      const double m1 = m[0] / h, m2 = m[1] / h;
      double q[2] = {0.0, 0.0};
      for (int t = sub; t < h; t += NSUB) {
        const double a = (double)xs[t * PT + p] - m1;
        const double b = (double)xs[(S - h + t) * PT + p] - m2;
        q[0] += a * a;
        q[1] += b * b;
      }
      column_sums<PT, 2>(q, red);
      const double e1 = m1 - mean, e2 = m2 - mean, em = (S & 1) ? mid - mean : 0.0;
      if (sub & 1) {
        if (h >= 2) {
          ag.add(m1, q[0] / (h - 1));
          ag.add(m2, q[1] / (h - 1));
        }
      } else {
        ag.add(mean, (q[0] + q[1] + h * (e1 * e1 + e2 * e2) + em * em) / (S - 1));
      }
    }
    if (t0 < t1) {
      // w[(u + j) % 16] holds the centred value at t + u + k0 + j
      auto at = [&](int r) { return r < S ? (double)xs[r * PT + p] - mean : 0.0; };
      double w[kDiagLpt];
#pragma unroll
      for (int j = 0; j < kDiagLpt - 1; ++j) w[j] = at(t0 + k0 + j);
      w[kDiagLpt - 1] = 0.0;
      int t = t0;
      // whole steps of 16 with every row in range for all lag groups
      const int tf = min(t1, S - klast - kDiagLpt);
      for (; t + kDiagLpt <= tf; t += kDiagLpt) {
        const float* pa = xs + t * PT + p;
        const float* pw = xs + (t + k0 + kDiagLpt - 1) * PT + p;
#pragma unroll
        for (int u = 0; u < kDiagLpt; ++u) {
          w[(u + kDiagLpt - 1) % kDiagLpt] = (double)pw[u * PT] - mean;
          const double a = (double)pa[u * PT] - mean;
#pragma unroll
          for (int j = 0; j < kDiagLpt; ++j) acc[j] = fma(a, w[(u + j) % kDiagLpt], acc[j]);
        }
      }
      for (; t < t1; t += kDiagLpt) {
#pragma unroll
        for (int u = 0; u < kDiagLpt; ++u) {
          w[(u + kDiagLpt - 1) % kDiagLpt] = at(t + u + k0 + kDiagLpt - 1);
          const double a = t + u < t1 ? (double)xs[(t + u) * PT + p] - mean : 0.0;
          if (t + u < t1)
#pragma unroll
            for (int j = 0; j < kDiagLpt; ++j) acc[j] = fma(a, w[(u + j) % kDiagLpt], acc[j]);
        }
      }
    }
  }
  // the segments' sums, in segment order
  __syncthreads();
  double* rs = reinterpret_cast<double*>(xs);  // [16][threads]
#pragma unroll
  for (int j = 0; j < kDiagLpt; ++j) rs[j * kDiagThreads + tid] = acc[j];
  __syncthreads();
  const int nl = kDiagPass * (int)gridDim.y;
  const size_t ldp = (size_t)nt * PT;
  for (int o = tid; o < kDiagPass * PT; o += kDiagThreads) {
    const int l = o / PT, pp = o % PT;
    double t = 0.0;
#pragma unroll
    for (int sg = 0; sg < NSEG; ++sg)
      t += rs[(l % kDiagLpt) * kDiagThreads + (sg * kDiagGroups + l / kDiagLpt) * PT + pp];
    gpart[((size_t)g * nl + kDiagPass * blockIdx.y + l) * ldp + (size_t)pos * PT + pp] = t;
  }
  if (stats && sub < 2) {
    const size_t st = (size_t)ng * ldp;
    double* a = agg + ((size_t)g * nt + pos) * PT + p + 3 * st * sub;
    a[0] = ag.mean_of_means;
    a[st] = ag.m2_of_means;
    a[2 * st] = ag.sum_var;
  }
}

// Per parameter, carried from one set of lags to the next.
struct DiagState {
  double tau, run, vw, ve;
};

// Advances the monotone sequence of a tile's parameters over the lags
// [base, base + nl) (the chain groups' sums added in group order), writes ess
// and, with the first lags, rhat; tiles with a parameter still positive and
// lags left go to next[0..*nnext).
template <int PT>
__global__ void __launch_bounds__(kDiagThreads)
diag_finish_kernel(const double* __restrict__ gpart, const double* __restrict__ agg, int C, int S,
                   int P, const int* __restrict__ tiles, int nt, int ng, int base, int nl,
                   DiagState* __restrict__ state, double* __restrict__ ess,
                   double* __restrict__ rhat, int* __restrict__ next, int* __restrict__ nnext) {
  __shared__ double rho[kDiagPass][PT];
  __shared__ double var[2][PT];  // var_within, var_estimator
  __shared__ int left, going;
  const int pos = blockIdx.x;
  const int tile = tiles ? tiles[pos] : pos;
  const int tid = threadIdx.x;
  const int p = tile * PT + tid;  // of the first PT threads
  const bool mine = tid < PT && p < P;
  const size_t ldp = (size_t)nt * PT;
  if (tid == 0) left = 0;
  DiagState s{};
  if (mine && base == 0) {
    ChainAgg full, split;
    const size_t st = (size_t)ng * ldp;
    const int h = S / 2;
    for (int g = 0; g < ng; ++g) {
      const double* a = agg + ((size_t)g * nt + pos) * PT + tid;
      const int n = diag_chain(C, g + 1, ng) - diag_chain(C, g, ng);
      full.merge(n, a[0], a[st], a[2 * st]);
      if (h >= 2) split.merge(2 * n, a[3 * st], a[4 * st], a[5 * st]);
    }
    s.tau = 0.0;
    s.run = INFINITY;
    full.stats(S, s.vw, s.ve);
    if (rhat) {
      double vw = 0.0, ve = 0.0;
      if (h >= 2) split.stats(h, vw, ve);
      rhat[p] = h >= 2 ? sqrt(ve / vw) : NAN;
    }
  } else if (mine) {
    s = state[p];
  }
  if (tid < PT) {
    var[0][tid] = s.vw;
    var[1][tid] = s.ve;
  }
  const int npair = S / 2;
  for (int b = 0; b < nl && (base + b) / 2 < npair; b += kDiagPass) {
    __syncthreads();
    if (tid == 0) going = 0;
    // rho_k = 1 - (var_within - mean_c gamma_ck) / var_estimator, rho_0 = 1
    for (int o = tid; o < kDiagPass * PT; o += kDiagThreads) {
      const int l = o / PT, pp = o % PT;
      const double* gp = gpart + (size_t)(b + l) * ldp + (size_t)pos * PT + pp;
      double t = 0.0;
#pragma unroll 8
      for (int g = 0; g < ng; ++g) t += gp[(size_t)g * nl * ldp];
      rho[l][pp] = base + b + l == 0 ? 1.0 : 1.0 - (var[0][pp] - t / S / (double)C) / var[1][pp];
    }
    __syncthreads();
    if (mine && s.run != 0.0) {
      // Rho_k = rho_2k + rho_2k+1; initial monotone sequence on Rho_1..
      for (int l = 0; l + 1 < kDiagPass; l += 2) {
        const int k = (base + b + l) / 2;
        if (k >= npair) break;
        double R = rho[l][tid] + rho[l + 1][tid];
        if (k >= 1) {
          R = R > 0.0 ? R : 0.0;
          s.run = R < s.run ? R : s.run;
          R = s.run;
        }
        s.tau += R;
        if (s.run == 0.0) break;  // the sequence stays at zero
      }
      if (s.run != 0.0) going = 1;
    }
    __syncthreads();
    if (!going) break;
  }
  if (mine) {
    ess[p] = (double)C * S / (-1.0 + 2.0 * s.tau);
    state[p] = s;
    if (s.run != 0.0 && (base + nl) / 2 < npair) left = 1;
  }
  __syncthreads();
  if (tid == 0 && left) next[atomicAdd(nnext, 1)] = tile;
}

__global__ void diag_zero_kernel(int* n) { *n = 0; }

constexpr int kDiagSlab = 1 << 18;

// Launch shape and workspace of one call.
struct DiagPlan {
  int pt, tiles, ng, cap;  // cap: workgroups resident on the chip
  int first;               // lag passes of the first round
  size_t agg, state, lists, part;  // bytes
  size_t total() const { return agg + state + lists + part; }
};

// PT: 32 parameters (128-byte rows) while a chain's tile leaves room for two
// workgroups per CU (S <= 608), narrower tiles for longer chains or few
// parameters.  The chains are split over as many groups as fill the chip
// twice.  More than kDiagSlab parameters are taken in slabs, which bounds the
// workspace.
static DiagPlan diag_plan(int C, int S, int P) {
  DiagPlan d{};
  constexpr int half = 160 * 1024 / 2 - 4096;  // LDS of a tile that lets two workgroups share a CU
  P = std::min(P, kDiagSlab);
  d.pt = S * 128 <= half && P > 16 ? 32 : S * 64 <= half && P > 8 ? 16 : 8;
  d.tiles = (P + d.pt - 1) / d.pt;
  d.cap = S * d.pt * 4 <= half ? 512 : 256;
  d.ng = std::max(1, std::min(C, 2 * d.cap / d.tiles));
  auto up = [](size_t b) { return (b + 255) / 256 * 256; };
  const size_t cols = (size_t)d.tiles * d.pt;
  d.agg = up(sizeof(double) * kAggDoubles * d.ng * cols);
  d.state = up(sizeof(DiagState) * (size_t)P);
  d.lists = up(sizeof(int) * (2 * (size_t)d.tiles + 2));
  // One round takes all lags of up to 256 draws where their workgroups fit the chip
  // at once: they run beside those of the first 32, and another round is three
  // launches, a copy and a wait (a call on 1 chain x 50, 100 and 200 draws of 60
  // parameters 47, 48 and 51 us in rounds, 36, 37 and 40 in one; 32, 39 and 53 with
  // a workgroup per parameter).  More draws leave the finish with more lags in a row
  // than rounds cost (4 x 1000 x 700 62 us, 102 in one).
  const int all = std::max(1, (S / 2 * 2 + kDiagPass - 1) / kDiagPass);
  d.first = all <= 8 && (int64_t)all * d.tiles * d.ng <= d.cap ? all : 1;
  // the first round, and room for more lags of the tiles that go on
  d.part = up(std::max(sizeof(double) * kDiagPass * d.first * d.ng * cols, (size_t)16 << 20));
  return d;
}

template <int PT>
static hipError_t diag_launch(const DiagPlan& d, const float* x, int C, int S, int P, int ldx,
                              double* ess, double* rhat, char* ws) {
  double* agg = reinterpret_cast<double*>(ws);
  DiagState* state = reinterpret_cast<DiagState*>(ws + d.agg);
  int* lists = reinterpret_cast<int*>(ws + d.agg + d.state);  // two lists, then the count
  double* part = reinterpret_cast<double*>(ws + d.agg + d.state + d.lists);
  int* count = lists + 2 * d.tiles;
  const size_t lds = std::max((size_t)S * PT * sizeof(float),
                              (size_t)kDiagLpt * kDiagThreads * sizeof(double));
  hipError_t e = hipFuncSetAttribute((const void*)diag_lags_kernel<PT>,
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return e;
  int nt = d.tiles, base = 0, passes = d.first;
  const int* list = nullptr;
  for (int it = 0;; ++it) {
    const int ng = it == 0 ? d.ng : std::max(1, std::min(C, 2 * d.cap / (nt * passes)));
    if (it > 0) {  // the most passes whose sums fit the workspace
      const size_t one = sizeof(double) * kDiagPass * ng * (size_t)nt * PT;
      passes = (int)std::max<size_t>(1, std::min<size_t>(passes, d.part / one));
    }
    const int fit = it == 0 ? ng
                            : (int)std::min<size_t>(ng, std::max<size_t>(
                                  1, d.part / (sizeof(double) * kDiagPass * passes * (size_t)nt * PT)));
    int* out = lists + (it & 1) * d.tiles;
    const bool last = (base + kDiagPass * passes) / 2 >= S / 2;  // no lags after these
    if (!last) hipLaunchKernelGGL(diag_zero_kernel, dim3(1), dim3(1), 0, 0, count);
    hipLaunchKernelGGL(diag_lags_kernel<PT>, dim3((nt * fit + 7) / 8 * 8, passes),
                       dim3(kDiagThreads), lds, 0, x, C, S, P, ldx, list, nt, fit, base, part,
                       it == 0 ? agg : nullptr);
    hipLaunchKernelGGL(diag_finish_kernel<PT>, dim3(nt), dim3(kDiagThreads), 0, 0, part, agg, C, S, P, list,
                       nt, fit, base, kDiagPass * passes, state, ess, rhat, out, count);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    base += kDiagPass * passes;
    int n = 0;
    if (!last) {
      e = hipMemcpyAsync(&n, count, sizeof(int), hipMemcpyDeviceToHost, 0);
      if (e != hipSuccess) return e;
    }
    e = hipStreamSynchronize(0);
    if (e != hipSuccess || n == 0) return e;
    nt = n;
    list = out;
    // lags per round grow, so that slowly mixing chains need few rounds
    passes = std::min(it == 0 ? 2 : 2 * passes, (2 * (S / 2) - base + kDiagPass - 1) / kDiagPass);
  }
}

}  // namespace nax

static int diag_check(const float* x, const double* ess, int chains, int draws, int params) {
  using namespace nax;
  if (!x || !ess || chains < 1 || draws < 2 || params < 1) {
    set_error("nax_diagnostics: need x, ess, chains >= 1, draws >= 2, params >= 1");
    return NAX_EINVAL;
  }
  if (draws > kDiagMaxDraws) {
    set_error("nax_diagnostics: at most 4096 draws per chain");
    return NAX_EINVAL;
  }
  return NAX_OK;
}

extern "C" int64_t nax_diagnostics_workspace(int32_t chains, int32_t draws, int32_t params) {
  if (chains < 1 || draws < 2 || params < 1 || draws > nax::kDiagMaxDraws) return 0;
  return (int64_t)nax::diag_plan(chains, draws, params).total();
}

extern "C" int nax_diagnostics_ws(const float* d_x, int32_t chains, int32_t draws, int32_t params,
                                  double* d_ess, double* d_split_rhat, void* d_ws,
                                  int64_t ws_bytes) {
  using namespace nax;
  const int rc = diag_check(d_x, d_ess, chains, draws, params);
  if (rc) return rc;
  const DiagPlan d = diag_plan(chains, draws, params);
  if (!d_ws || ws_bytes < (int64_t)d.total() || reinterpret_cast<uintptr_t>(d_ws) % 256) {
    set_error("nax_diagnostics_ws: need a 256-byte aligned workspace of "
              "nax_diagnostics_workspace() bytes");
    return NAX_EINVAL;
  }
  char* ws = static_cast<char*>(d_ws);
  for (int64_t p = 0; p < params; p += kDiagSlab) {
    const int n = (int)std::min<int64_t>(kDiagSlab, params - p);
    double* rh = d_split_rhat ? d_split_rhat + p : nullptr;
    DiagPlan ds = d;
    ds.tiles = (n + d.pt - 1) / d.pt;
    const auto go = d.pt == 32 ? diag_launch<32> : d.pt == 16 ? diag_launch<16> : diag_launch<8>;
    const hipError_t e = go(ds, d_x + p, chains, draws, n, params, d_ess + p, rh, ws);
    if (e != hipSuccess) {
      set_error(std::string("nax_diagnostics: ") + hipGetErrorString(e));
      return NAX_EHIP;
    }
  }
  return NAX_OK;
}

extern "C" int nax_diagnostics(const float* d_x, int32_t chains, int32_t draws, int32_t params,
                               double* d_ess, double* d_split_rhat) {
  using namespace nax;
  const int rc = diag_check(d_x, d_ess, chains, draws, params);
  if (rc) return rc;
  const size_t bytes = diag_plan(chains, draws, params).total();
  void* ws = nullptr;
  const hipError_t e = hipMalloc(&ws, bytes);
  if (e != hipSuccess) {
    set_error(std::string("nax_diagnostics: workspace: ") + hipGetErrorString(e));
    return NAX_ENOMEM;
  }
  const int out = nax_diagnostics_ws(d_x, chains, draws, params, d_ess, d_split_rhat, ws,
                                     (int64_t)bytes);
  (void)hipFree(ws);
  return out;
}
