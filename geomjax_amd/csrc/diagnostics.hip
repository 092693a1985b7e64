// Multi-chain effective sample size and potential scale reduction of a
// [T, C, D] sample array on the device (float64 arithmetic).
//
// Reference: geomjax/diagnostics.py:25-75 (potential_scale_reduction) and
// :78-209 (effective_sample_size: autocovariance of every chain, the
// mean autocovariance over chains, Geyer's initial positive and initial
// monotone sequences, tau floored at 1 / log10(M N)).  The reference forms
// the autocovariances by FFT with zero padding to at least 2N; that is the
// same quantity as the direct sums taken here,
//   acov_c(k) = (1/N) sum_{t < N-k} (x_{t,c} - m_c)(x_{t+k,c} - m_c),
// which for the sample windows of this path (N up to a few thousand) cost
// less than a transform.
//
// Pass 1 (lag_block_kernel, series up to kBlockMaxN with at least kBlockMinLanes coordinates
// or chains): a lane holds one series.  Its 64 lanes are 64 coordinates of a
// chain (or 64 chains of a coordinate when coordinates are few), the centred series
// lie in LDS as [sample][lane] in float64, and each of the four waves sums eight
// consecutive lags at a time with a window of eight values in registers: two LDS reads
// per eight FMAs.  Workgroups are (chain tile, 64 lanes, 32 lags); the chains of a
// tile are added in order.  Bound: float64 FMAs and the LDS reads about alike.
// The form before (lag_sums_kernel: thread k sums lag k, two LDS reads per FMA,
// 100 of 256 lanes busy at 100 samples, each 4-byte load from a line of its own) took
// 870 us at 100 x 4096 x 64 float32; this one 240 us (42 us for R-hat alone).  It stays for longer series and for few
// series, where a thread per lag is the only parallelism.  Without an ESS
// (R-hat alone) only means and variances are formed.
// Pass 2, one workgroup per coordinate: the tiles' sums are added, the correlations
// formed in parallel, and one lane runs the sequential Geyer steps on LDS (at
// most N/2 of them).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "../../include/geomjax_amd.h"
#include "common.h"

namespace gjx {
namespace diag {

constexpr int kMaxTile = 16;  // chains per pass-1 workgroup at most
constexpr int kThreads = 256;
constexpr size_t kLdsBytes = 160 * 1024 - 1024;  // dynamic LDS of pass 1 at most

// chains per pass-1 workgroup for series of length N (0: too long)
__host__ __device__ inline int tile_chains(int N) {
  const size_t t = kLdsBytes / ((size_t)N * sizeof(double));
  return (int)(t < (size_t)kMaxTile ? t : (size_t)kMaxTile);
}

template <class T>
__global__ void __launch_bounds__(kThreads) lag_sums_kernel(const T* __restrict__ x, int N, int C, int tc,
                                                            int64_t st, int64_t sc, int64_t sd,
                                                            double* __restrict__ lag, double* __restrict__ cmean,
                                                            double* __restrict__ cvar) {
  extern __shared__ double xs[];  // [tc][N] centred series
  const int d = blockIdx.y, tile = blockIdx.x, D = gridDim.y;
  const int c0 = tile * tc;
  const int nc = min(tc, C - c0);
  const int tid = threadIdx.x;
  __shared__ double red[kMaxTile][kThreads / 64];
  // load the tile's series and their means
  for (int j = 0; j < nc; ++j) {
    double s = 0.0;
    for (int t = tid; t < N; t += kThreads) {
      const double v = (double)x[(int64_t)t * st + (int64_t)(c0 + j) * sc + (int64_t)d * sd];
      xs[j * N + t] = v;
      s += v;
    }
    s = group_sum<64>(s);
    if (tid % 64 == 0) red[j][tid / 64] = s;
  }
  __syncthreads();
  for (int j = 0; j < nc; ++j) {
    const double m = (red[j][0] + red[j][1] + red[j][2] + red[j][3]) / (double)N;
    for (int t = tid; t < N; t += kThreads) xs[j * N + t] -= m;
    if (tid == 0) cmean[(int64_t)d * C + c0 + j] = m;
  }
  __syncthreads();
  // lag sums over the tile's chains
  for (int k = tid; k < N; k += kThreads) {
    double s = 0.0;
    for (int j = 0; j < nc; ++j) {
      const double* a = xs + j * N;
      for (int t = 0; t + k < N; ++t) s = fma(a[t], a[t + k], s);
    }
    lag[((int64_t)tile * D + d) * N + k] = s;
  }
  // per-chain variance (unbiased), for R-hat
  for (int j = 0; j < nc; ++j) {
    double s = 0.0;
    for (int t = tid; t < N; t += kThreads) s = fma(xs[j * N + t], xs[j * N + t], s);
    s = group_sum<64>(s);
    __syncthreads();
    if (tid % 64 == 0) red[j][tid / 64] = s;
    __syncthreads();
    if (tid == 0) cvar[(int64_t)d * C + c0 + j] = (red[j][0] + red[j][1] + red[j][2] + red[j][3]) / (double)(N - 1);
  }
}

constexpr int kLags = 8;                 // lags per wave
constexpr int kGroup = kLags * kThreads / 64;  // lags per workgroup
constexpr int kPad = 2 * kLags;          // zero rows after the series (the window reads past its end)
constexpr int kRow = 65;                 // doubles per row of the staged series (64 lanes)
constexpr int kBlockMaxN = (int)(kLdsBytes / (kRow * sizeof(double))) - kPad - 8;
constexpr int kBlockMinLanes = 32;

// Lag sums, means and variances of the series of one (chain tile, 64 lanes).  LANE_D:
// the lanes are coordinates d0 .. d0 + 63 and the tile's chains are taken in
// turn; else the lanes are chains of coordinate blockIdx.y, 64 at a time, and
// the lag sums are added over the lanes at the end.
template <class T, bool LANE_D>
__global__ void __launch_bounds__(kThreads) lag_block_kernel(const T* __restrict__ x, int N, int C, int D, int tc,
                                                             int64_t st, int64_t sc, int64_t sd, bool want_lags,
                                                             double* __restrict__ lag, double* __restrict__ cmean,
                                                             double* __restrict__ cvar) {
  extern __shared__ double ys[];  // [N + kPad][kRow]
  __shared__ double part[2][kThreads / 64][64];
  const int tid = threadIdx.x, l = tid % 64, w = __builtin_amdgcn_readfirstlane(tid / 64);
  const int c0 = blockIdx.x * tc, nc = min(tc, C - c0);
  const int k0 = ((int)blockIdx.z * (kThreads / 64) + w) * kLags;
  const bool outer = blockIdx.z == 0;  // this workgroup writes the means and variances
  for (int i = tid; i < kPad * kRow; i += kThreads) ys[N * kRow + i] = 0.0;
  double acc[kLags];
#pragma unroll
  for (int j = 0; j < kLags; ++j) acc[j] = 0.0;
  const int rounds = LANE_D ? nc : (nc + 63) / 64;
  for (int it = 0; it < rounds; ++it) {
    // stage 64 series; lanes past the last one hold zeros
    const int c = LANE_D ? c0 + it : c0 + 64 * it + l;
    const int d = LANE_D ? (int)blockIdx.y * 64 + l : (int)blockIdx.y;
    const bool ok = LANE_D ? d < D : c < c0 + nc;
    const T* const xs = x + (ok ? (int64_t)c * sc + (int64_t)d * sd : 0);
    double s = 0.0;
    // eight loads in flight a lane (one at a time, their latency was most of the pass)
    for (int t0 = w; t0 < N; t0 += 8 * (kThreads / 64)) {
      T v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = xs[(int64_t)min(t0 + e * (kThreads / 64), N - 1) * st];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int t = t0 + e * (kThreads / 64);
        if (t < N) {
          const double y = ok ? (double)v[e] : 0.0;
          ys[t * kRow + l] = y;
          s += y;
        }
      }
    }
    part[0][w][l] = s;
    __syncthreads();
    const double m = (part[0][0][l] + part[0][1][l] + part[0][2][l] + part[0][3][l]) / (double)N;
    double q = 0.0;
#pragma unroll 4
    for (int t = w; t < N; t += kThreads / 64) {
      const double v = ys[t * kRow + l] - m;
      ys[t * kRow + l] = v;
      q = fma(v, v, q);
    }
    part[1][w][l] = q;
    __syncthreads();
    if (outer && ok && w == 0) {
      cmean[(int64_t)d * C + c] = m;
      cvar[(int64_t)d * C + c] = (part[1][0][l] + part[1][1][l] + part[1][2][l] + part[1][3][l]) / (double)(N - 1);
    }
    if (want_lags && k0 < N) {
      const double* const a = ys + l;
      double win[kLags];  // samples t + k0 .. t + k0 + 7, sample t + k0 + j in slot (t + j) % 8
#pragma unroll
      for (int j = 0; j < kLags; ++j) win[j] = a[(k0 + j) * kRow];
      for (int t = 0; t < N - k0; t += kLags) {
#pragma unroll
        for (int u = 0; u < kLags; ++u) {
          const double y = a[(t + u) * kRow];
#pragma unroll
          for (int j = 0; j < kLags; ++j) acc[j] = fma(y, win[(u + j) % kLags], acc[j]);
          win[u] = a[(t + u + k0 + kLags) * kRow];
        }
      }
    }
    __syncthreads();
  }
  if (!want_lags || k0 >= N) return;
  const int tile = blockIdx.x;
  if constexpr (LANE_D) {
    const int d = (int)blockIdx.y * 64 + l;
    if (d < D) {
      double* const out = lag + ((int64_t)tile * D + d) * N + k0;
#pragma unroll
      for (int j = 0; j < kLags; ++j)
        if (k0 + j < N) out[j] = acc[j];
    }
  } else {
    double* const out = lag + ((int64_t)tile * D + blockIdx.y) * N + k0;
#pragma unroll
    for (int j = 0; j < kLags; ++j) {
      const double t = group_sum<64>(acc[j]);
      if (l == 0 && k0 + j < N) out[j] = t;
    }
  }
}

// Sum of v over the workgroup (kThreads lanes), identical in every lane.
__device__ double block_sum(double v, double* sh) {
  v = group_sum<64>(v);
  __syncthreads();
  if (threadIdx.x % 64 == 0) sh[threadIdx.x / 64] = v;
  __syncthreads();
  double t = 0.0;
  for (int w = 0; w < kThreads / 64; ++w) t += sh[w];
  __syncthreads();
  return t;
}

constexpr int kRhoLds = 4096;  // correlations of series up to this length stay in LDS

__global__ void __launch_bounds__(kThreads) finalize_kernel(const double* __restrict__ lag,
                                                            const double* __restrict__ cmean,
                                                            const double* __restrict__ cvar, int N, int C,
                                                            int ntiles, double* __restrict__ rho,
                                                            double* __restrict__ ess, double* __restrict__ rhat) {
  const int d = blockIdx.x, D = gridDim.x, tid = threadIdx.x;
  __shared__ double sh[kThreads / 64];
  __shared__ double rs[kRhoLds];
  double* r = N <= kRhoLds ? rs : rho + (int64_t)d * N;  // mean autocovariance, then rho
  if (ess) {
    // kP threads per lag when lags are few, each with its share of the tiles
    const int P = N <= kThreads / 8 ? 8 : (N <= kThreads / 4 ? 4 : (N <= kThreads / 2 ? 2 : 1));
    const int64_t step = (int64_t)D * N;
    for (int k = tid / P; k < N; k += kThreads / P) {
      double s = 0.0;
      const double* p = lag + (int64_t)d * N + k;
#pragma unroll 8
      for (int tl = tid % P; tl < ntiles; tl += P) s += p[tl * step];
      if (P >= 2) s += dpp<0xB1>(s);
      if (P >= 4) s += dpp<0x4E>(s);
      if (P >= 8) s += dpp<0x141>(s);
      if (tid % P == 0) r[k] = s / ((double)N * (double)C);
    }
  }
  // variance of the chain means (unbiased) and the mean within-chain variance
  double sm = 0.0, sv = 0.0;
  for (int c = tid; c < C; c += kThreads) {
    sm += cmean[(int64_t)d * C + c];
    sv += cvar[(int64_t)d * C + c];
  }
  const double mbar = block_sum(sm, sh) / (double)C;
  const double within = block_sum(sv, sh) / (double)C;
  double sq = 0.0;
  for (int c = tid; c < C; c += kThreads) {
    const double e = cmean[(int64_t)d * C + c] - mbar;
    sq = fma(e, e, sq);
  }
  const double var_means = block_sum(sq, sh) / (double)(C - 1);
  if (rhat && tid == 0) rhat[d] = sqrt(((double)N * var_means / within + (double)N - 1.0) / (double)N);
  if (!ess) return;
  __syncthreads();
  // Geyer's initial positive and initial monotone sequences (diagnostics.py:150-209)
  const double var0 = r[0] * (double)N / ((double)N - 1.0);
  const double weighted_var = var0 * ((double)N - 1.0) / (double)N + var_means;
  const int n_even = N - N % 2, K = n_even / 2;
  __syncthreads();  // every lane has read r[0]
  for (int k = tid; k < n_even; k += kThreads) r[k] = k == 0 ? 1.0 : 1.0 - (var0 - r[k]) / weighted_var;
  __syncthreads();
  if (tid != 0) return;
  // rho_even[i] = r[2i], rho_odd[i] = r[2i + 1]; mask = positive pair sums so far
  int count = 0;
  bool all_pos = true;
  for (int i = 0; i < K; ++i) {
    all_pos = all_pos && (r[2 * i] + r[2 * i + 1] > 0.0);
    if (all_pos) ++count;
  }
  const int max_t = count > 0 ? count - 1 : 0;
  const int idx = max_t + 1;
  const bool in_range = idx < K;
  const int idc = idx < K ? idx : K - 1;
  const double gathered = r[2 * idc];
  double sum = 0.0, running = 0.0, last_even_f = 0.0;
  for (int i = 0; i < K; ++i) {
    const bool m = i < count;  // the mask is a prefix
    const bool me = (in_range && i == idx) ? (gathered > 0.0) : m;
    const double re = me ? r[2 * i] : 0.0;
    const double ro = m ? r[2 * i + 1] : 0.0;
    const double s = re + ro;
    const double prev = i == 0 ? s : running;
    running = i == 0 ? s : fmin(running, s);
    const bool update = s > prev;
    const double ref = update ? running / 2.0 : re;
    const double rof = update ? running / 2.0 : ro;
    sum += ref + rof;
    if (i == idc) last_even_f = ref;
  }
  double tau = -1.0 + 2.0 * sum - last_even_f;
  tau = fmax(tau, 1.0 / log10((double)C * (double)N));
  ess[d] = (double)C * (double)N / tau;
}

}  // namespace diag

int diagnostics_max_samples() { return (int)(diag::kLdsBytes / sizeof(double)); }

uint64_t diagnostics_workspace_bytes(int N, int C, int D) {
  const int tc = diag::tile_chains(N);
  const int64_t ntiles = (C + tc - 1) / tc;
  return (uint64_t)(ntiles * D * N + 2 * (int64_t)D * C + (int64_t)D * N) * sizeof(double);
}

hipError_t launch_diagnostics(const void* x, int dtype, int N, int C, int D, int64_t st, int64_t sc, int64_t sd,
                              void* workspace, double* ess, double* rhat, hipStream_t stream) {
  const int tc = diag::tile_chains(N);
  int ntiles = (C + tc - 1) / tc;
  double* lag = static_cast<double*>(workspace);
  double* cmean = lag + (int64_t)ntiles * D * N;
  double* cvar = cmean + (int64_t)D * C;
  double* rho = cvar + (int64_t)D * C;
  // Lanes along coordinates read whole lines of [sample, chain, coordinate] arrays, but a
  // workgroup then takes its tile's chains in turn: only when the tiles fill the
  // chip twice (or there are too few chains for lanes along them).
  const int64_t groups = ess != nullptr ? (N + diag::kGroup - 1) / diag::kGroup : 1;
  const bool lane_d = D >= diag::kBlockMinLanes &&
                      (ess == nullptr || (int64_t)ntiles * ((D + 63) / 64) * groups >= 512 || C < diag::kBlockMinLanes);
  auto run = [&](auto zero) -> hipError_t {
    using T = decltype(zero);
    const T* p = static_cast<const T*>(x);
    if (N <= diag::kBlockMaxN && (lane_d || C >= diag::kBlockMinLanes)) {
      const size_t lds = (size_t)(N + diag::kPad) * diag::kRow * sizeof(double);
      const bool lags = ess != nullptr;
      auto k = lane_d ? diag::lag_block_kernel<T, true> : diag::lag_block_kernel<T, false>;
      // chains per workgroup: a tile as the partial sums are laid out (without lag sums there
      // are none: a few), or one for each lane (fewer workgroups than tiles)
      static_assert(diag::kMaxTile <= 64, "64 chains a workgroup need no more partial sums than tiles");
      const int per = !lane_d ? 64 : lags ? tc : std::max(1, C / 1024);
      ntiles = (C + per - 1) / per;
      hipError_t e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      if (e != hipSuccess) return e;
      const dim3 g((unsigned)ntiles, lane_d ? (unsigned)((D + 63) / 64) : (unsigned)D, (unsigned)groups);
      hipLaunchKernelGGL(k, g, dim3(diag::kThreads), lds, stream, p, N, C, D, per, st, sc, sd, lags, lag, cmean, cvar);
      return hipSuccess;
    }
    const size_t lds = (size_t)tc * N * sizeof(double);
    auto k = diag::lag_sums_kernel<T>;
    hipError_t e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k, dim3((unsigned)ntiles, (unsigned)D), dim3(diag::kThreads), lds, stream, p, N, C, tc, st, sc,
                       sd, lag, cmean, cvar);
    return hipSuccess;
  };
  hipError_t e = dtype == GJX_F32 ? run(0.0f) : run(0.0);
  if (e != hipSuccess) return e;
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(diag::finalize_kernel, dim3((unsigned)D), dim3(diag::kThreads), 0, stream, lag, cmean, cvar, N,
                     C, ntiles, rho, ess, rhat);
  return hipGetLastError();
}

}  // namespace gjx
