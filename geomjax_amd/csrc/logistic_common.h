// Device routines of the float64 logistic-regression kernels (Fisher metric):
// LDS layout, passes over X with MFMA Gram / quadratic forms, the symmetric
// sweep inverse and the Cholesky used for momentum draws.
//
// One workgroup of NT = 256 lanes (4 waves) per chain.  Everything is
// parameterised by the feature capacity MD (64 or 128) through Cfg<MD>:
//   TB 16-wide tiles per dimension, NLT lower tiles of the Gram, BS the BS x BS
//   block of the inverse each lane holds during the sweep (16 x 16 lanes cover
//   the matrix), LDX the padded LDS row stride of the matrix.
//
// Passes over X.  Each wave takes whole 16-row blocks (block w, w + 4, ...) and
// reads them from global memory (L2: all chains of a posterior share X) straight
// into the operand layout of v_mfma_f64_16x16x4f64, so the loops hold no barrier
// and no LDS staging; the waves' partial sums meet in LDS once per pass.  Bound:
// the float64 matrix pipe, 64 cycles an MFMA and 40 MFMAs per 16 rows and pass at
// D = 64 (40 us a pass and workgroup at 2.07 GHz), plus the passes' own VALU
// instructions, which do not overlap float64 MFMAs (measured: 4 cycles added
// per instruction, float32 ones too).  At 2048 x 64 with two workgroups on a CU a
// Gram pass takes 50 us, a quadratic-form pass 51, a sweep 12 per workgroup.  The
// form before (32-row chunks of X staged in LDS behind four barriers each, the
// tiles dealt to the waves 3, 3, 2, 2, 64 MFMAs per 16 rows in the second
// pass) made a transition of 1024 chains, 10 steps, 107.5 ms; this one 30.7 ms.
#pragma once

#include <type_traits>

#include "common.h"
#include "logistic_tiles.h"

namespace gjx {
namespace logistic {

// The lane's index in the workgroup, opaque to the compiler: addresses formed from it
// inside a pass are not hoisted above the stage loop of a chain, where they only spill.
// At capacity 64 the RMHMC loop spilled 157 registers without it and 84 with it (2048 x 64,
// 1024 chains: 30.7 -> 30.3 ms), MMALA 159 and 86 (four transitions: 5.68 -> 5.46 ms).
__device__ __forceinline__ int pass_thread() {
  int t = (int)threadIdx.x;
  asm volatile("" : "+v"(t));
  return t;
}

constexpr int NT = 256;

template <int MD>
struct Cfg {
  static_assert(MD == 64 || MD == 128, "feature capacity 64 or 128");
  static constexpr int MAXD = MD;
  static constexpr int LDX = MD + 1;
  static constexpr int TB = MD / 16;
  static constexpr int NLT = TB * (TB + 1) / 2;
  static constexpr int BS = MD / 16;
  // Gram pass: the waves form H groups, each with its share of the tiles (288
  // registers of tiles at 128 features do not leave room for the rows)
  static constexpr int H = MD == 64 ? 1 : 2;
};

typedef double f64x4 __attribute__((ext_vector_type(4)));

template <class C>
struct Smem {
  union {
    double Gi[C::MAXD * C::LDX];        // G, then the Cholesky factor or G^-1
    double tile[2 * (C::NLT / C::H) * 256];  // two waves' partial Gram tiles at the end of a Gram pass
  };
  double rowbuf[2][C::MAXD];  // sweep: the pivot row
  double part[4][C::MAXD];    // the waves' partial sums of X^T r, X^T h, G v
  double dk[C::MAXD];         // pivots of the last sweep
  double q0[C::MAXD], p0[C::MAXD], q[C::MAXD], p[C::MAXD], u[C::MAXD], dH[C::MAXD], g[C::MAXD], z[C::MAXD],
      qs[C::MAXD];
  double gv[C::MAXD], vt[C::MAXD];
  double red[8];
};

template <class C>
__device__ __forceinline__ double block_sum(Smem<C>& S, double v) {
  v = group_sum<64>(v);
  const int w = threadIdx.x / 64, l = threadIdx.x % 64;
  __syncthreads();
  if (l == 0) S.red[w] = v;
  __syncthreads();
  return S.red[0] + S.red[1] + S.red[2] + S.red[3];
}

template <class C>
__device__ __forceinline__ double block_max(Smem<C>& S, double v) {
  v = group_reduce<64, NanMax>(v);
  const int w = threadIdx.x / 64, l = threadIdx.x % 64;
  __syncthreads();
  if (l == 0) S.red[w] = v;
  __syncthreads();
  return nan_max(nan_max(S.red[0], S.red[1]), nan_max(S.red[2], S.red[3]));
}

__device__ __forceinline__ double softplus(double x) { return fmax(x, 0.0) + log1p(exp(-fabs(x))); }
__device__ __forceinline__ double sigmoid(double x) { return 1.0 / (1.0 + exp(-x)); }

// Sum over the four 16-lane rows of the wave (lanes l, l ^ 16, l ^ 32, l ^ 48),
// the same in all four.
__device__ __forceinline__ double rows_sum(double v) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const auto lo = __builtin_amdgcn_permlane16_swap((uint32_t)b, (uint32_t)b, false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap((uint32_t)(b >> 32), (uint32_t)(b >> 32), false, false);
  const double s = __builtin_bit_cast(double, ((uint64_t)hi[0] << 32) | lo[0]) +
                   __builtin_bit_cast(double, ((uint64_t)hi[1] << 32) | lo[1]);
  const uint64_t c = __builtin_bit_cast(uint64_t, s);
  const auto lo2 = __builtin_amdgcn_permlane32_swap((uint32_t)c, (uint32_t)c, false, false);
  const auto hi2 = __builtin_amdgcn_permlane32_swap((uint32_t)(c >> 32), (uint32_t)(c >> 32), false, false);
  return __builtin_bit_cast(double, ((uint64_t)hi2[0] << 32) | lo2[0]) +
         __builtin_bit_cast(double, ((uint64_t)hi2[1] << 32) | lo2[1]);
}

// Sums of four values over the 16 lanes of a row, one per lane: lane l receives
// the total of e[l % 4] (the four lanes with that l % 4 the same bits).
__device__ __forceinline__ double sum4_of_16(const double (&e)[4], int l) {
  const bool b0 = l & 1, b1 = l & 2;
  const double k0 = (b0 ? e[1] : e[0]) + dpp<0xB1>(b0 ? e[0] : e[1]);
  const double k1 = (b0 ? e[3] : e[2]) + dpp<0xB1>(b0 ? e[2] : e[3]);
  double v = (b1 ? k1 : k0) + dpp<0x4E>(b1 ? k0 : k1);
  v += dpp<0x128>(v);         // row_ror 8
  return v + dpp<0x124>(v);  // row_ror 4
}

// v of lane J of each quad
template <int J>
__device__ __forceinline__ double quad_bcast(double v) { return dpp<J * 0x55>(v); }

// Gram pass at S.q: S.Gi = X^T diag(lambda + coef w (X vec)) X + I / prior_var
// (vec == nullptr: the Fisher metric G itself) in the first D rows and columns
// (nothing meaningful past them: load_block reads zeros there).  With want_lg it
// also returns the log-likelihood sum and leaves grad l = X^T (y - s) - q/prior_var
// in S.g; with want_gv it leaves G vec = X^T (lambda (X vec)) + vec/prior_var in
// S.gv.  S.q and vec are zero past D over the capacity.
//
// NB = ceil(D / 16) feature tiles.  Lane l = 16 g + m holds X[n0 + 4 j + g][16 b + m]
// (j < 4, b < NB) of a 16-row block: for each j both operands of the K step of rows
// 4 j .. 4 j + 3.  eta of the lane's row n0 + 4 (l % 4) + g comes from a reduce-scatter
// over the 16 lanes, so the sigmoid is evaluated once per row and four lanes; the
// weight of K step j is lane j's of each quad.
// Tiles T0 .. T0 + NT of the lower triangle, for the wave's share of the rows: blocks
// w, w + WR, ...
template <class C, int NB, int T0, int NTW, bool VEC, bool LG>
__device__ __forceinline__ void gram_loop(Smem<C>& S, const double* X, const double* y, int N, int D, const double* vec,
                                          double coef, bool want_gv, int w, f64x4 (&acc)[NTW], double& ll,
                                          double (&gacc)[NB], double (&gvacc)[NB]) {
  constexpr int WR = 4 / C::H;
  const int l = pass_thread() % 64;
  const int g = l / 16, m = l % 16;
  const int nblk = (N + 15) / 16;
  if (nblk == 0) return;
  double qv[NB], vv[VEC ? NB : 1];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    qv[b] = S.q[16 * b + m];
    if constexpr (VEC) vv[b] = vec[16 * b + m];
  }
  struct Blk {
    double x[4][NB];
    double y;
  };
  // features past D, all in the last tile, read feature D - 1 and rows past N row
  // N - 1 (in bounds; they meet zeros or tile entries that are not used); past its
  // last block a wave re-reads the last one with weights of zero
  // (byte offsets from a block's first row: a uniform base, one 32-bit lane offset
  // per K step and immediate offsets per tile)
  const uint32_t mb = 8u * (uint32_t)m, lastb = last_tile_bytes(NB, m, D);
  uint32_t rowb[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) rowb[j] = 8u * (uint32_t)((4 * j + g) * D);
  auto fetch_row = [&](Blk& B, int blk, int j) {
    const int n0 = 16 * min(blk, nblk - 1);
    const char* const Xb = reinterpret_cast<const char*>(X + (size_t)n0 * D);
    const uint32_t row = row_bytes(rowb[j], n0, N, D);
    const double* const xr = reinterpret_cast<const double*>(Xb + (row + mb));
#pragma unroll
    for (int b = 0; b < NB - 1; ++b) B.x[j][b] = xr[16 * b];
    B.x[j][NB - 1] = *reinterpret_cast<const double*>(Xb + (row + lastb));
  };
  auto fetch_y = [&](Blk& B, int blk) {
    const int n0 = 16 * min(blk, nblk - 1);
    if constexpr (LG) B.y = (y + n0)[min(4 * (l & 3) + g, N - n0 - 1)];
  };
  struct Wt {
    double lam, rr, bb;
  };
  auto weights = [&](const Blk& B, int blk, Wt& o) {
    double e[4], v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      e[j] = 0.0;
      v[j] = 0.0;
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        e[j] = fma(B.x[j][b], qv[b], e[j]);
        if constexpr (VEC) v[j] = fma(B.x[j][b], vv[b], v[j]);
      }
    }
    const double eta = sum4_of_16(e, l);
    const bool ok = 16 * blk + 4 * (l & 3) + g < N;
    const double s = sigmoid(eta);
    const double lam = s * (1.0 - s);
    o.lam = ok ? lam : 0.0;
    if constexpr (VEC) {
      const double xv = sum4_of_16(v, l);
      o.lam = ok ? lam + coef * lam * (1.0 - 2.0 * s) * xv : 0.0;
      o.bb = ok ? lam * xv : 0.0;
    }
    if constexpr (LG) {
      o.rr = ok ? B.y - s : 0.0;
      if (ok && m < 4) ll += B.y * eta - softplus(eta);
    }
  };
  auto kstep = [&](const Blk& B, const Wt& o, auto jc) {
    constexpr int j = decltype(jc)::value;
    const double lm = quad_bcast<j>(o.lam);
    double xl[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) xl[b] = lm * B.x[j][b];
    int t = 0;
#pragma unroll
    for (int bi = 0; bi < NB; ++bi)
#pragma unroll
      for (int bj = 0; bj <= bi; ++bj) {
        if (t >= T0 && t < T0 + NTW)
          acc[t - T0] = __builtin_amdgcn_mfma_f64_16x16x4f64(xl[bi], B.x[j][bj], acc[t - T0], 0, 0, 0);
        ++t;
      }
    if constexpr (LG) {
      const double r = quad_bcast<j>(o.rr);
#pragma unroll
      for (int b = 0; b < NB; ++b) gacc[b] = fma(B.x[j][b], r, gacc[b]);
    }
    if constexpr (VEC) {
      if (want_gv) {
        const double r = quad_bcast<j>(o.bb);
#pragma unroll
        for (int b = 0; b < NB; ++b) gvacc[b] = fma(B.x[j][b], r, gvacc[b]);
      }
    }
  };
  // One register set: each K step's rows are reloaded for the next block as soon
  // as its MFMAs are issued (the scheduling barriers keep the loads there: hoisted,
  // they need a second set and spill); the second wave of the SIMD covers the
  // latency of the last ones.
  Blk B;
  Wt o;
  auto kstep_and_reload = [&](int blk, auto jc) {
    kstep(B, o, jc);
    __builtin_amdgcn_sched_barrier(0);
    fetch_row(B, blk + WR, decltype(jc)::value);
  };
#pragma unroll
  for (int j = 0; j < 4; ++j) fetch_row(B, w, j);
  fetch_y(B, w);
  weights(B, w, o);
  for (int blk = w; blk < nblk; blk += WR) {
    fetch_y(B, blk + WR);
    kstep_and_reload(blk, std::integral_constant<int, 0>{});
    kstep_and_reload(blk, std::integral_constant<int, 1>{});
    kstep_and_reload(blk, std::integral_constant<int, 2>{});
    kstep_and_reload(blk, std::integral_constant<int, 3>{});
    weights(B, blk + WR, o);
  }
}

template <class C, int NB, bool VEC, bool LG>
__device__ __forceinline__ void gram_pass_nb(Smem<C>& S, const double* X, const double* y, int N, int D, double prior_var,
                                             const double* vec, double coef, bool want_gv, double& loglik) {
  constexpr int NTL = NB * (NB + 1) / 2, NTW = (NTL + C::H - 1) / C::H;
  const int t = pass_thread(), l = t % 64, w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64);
  f64x4 acc[NTW];
#pragma unroll
  for (int i = 0; i < NTW; ++i) acc[i] = f64x4{0, 0, 0, 0};
  double ll = 0.0, gacc[NB], gvacc[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) gacc[b] = gvacc[b] = 0.0;
  if constexpr (C::H == 1) {
    gram_loop<C, NB, 0, NTW, VEC, LG>(S, X, y, N, D, vec, coef, want_gv, w, acc, ll, gacc, gvacc);
  } else {
    // the likelihood and the vector sums belong to the first group
    if (w < 2) {
      gram_loop<C, NB, 0, NTW, VEC, LG>(S, X, y, N, D, vec, coef, want_gv, w, acc, ll, gacc, gvacc);
    } else {
      gram_loop<C, NB, NTW, NTW, VEC, false>(S, X, y, N, D, vec, coef, false, w - 2, acc, ll, gacc, gvacc);
    }
  }
  // the partial tiles of a group's waves meet in its first wave, through LDS
  auto put = [&](double* P) {
#pragma unroll
    for (int i = 0; i < NTW; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) P[(i * 4 + r) * 64 + l] = acc[i][r];
  };
  auto add = [&](const double* P) {
#pragma unroll
    for (int i = 0; i < NTW; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][r] += P[(i * 4 + r) * 64 + l];
  };
  // both triangles of G from lower tiles T0 .., C[4r + l/16][l%16] layout
  auto store = [&](auto t0c) {
    constexpr int T0 = decltype(t0c)::value;
    int i0 = 0;
#pragma unroll
    for (int bi = 0; bi < NB; ++bi)
#pragma unroll
      for (int bj = 0; bj <= bi; ++bj) {
        if (i0 >= T0 && i0 < T0 + NTW) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int i = bi * 16 + 4 * r + l / 16, j = bj * 16 + l % 16;
            // a diagonal tile holds (i, j) and (j, i) rounded differently: keep the
            // lower one for both so that G is exactly symmetric
            if (i < j) continue;
            const double a = acc[i0 - T0][r];
            const double v = i == j ? a + 1.0 / prior_var : a;
            S.Gi[i * C::LDX + j] = v;
            S.Gi[j * C::LDX + i] = v;
          }
        }
        ++i0;
      }
  };
  if (LG) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const double s = rows_sum(gacc[b]);
      if (l < 16) S.part[w][16 * b + l] = s;
    }
  }
  __syncthreads();
  if constexpr (C::H == 1) {
    if (w >= 2) put(S.tile + (w - 2) * (NTW * 256));
    __syncthreads();
    if (w < 2) add(S.tile + w * (NTW * 256));
    __syncthreads();
    if (w == 1) put(S.tile);
  } else {
    if (w & 1) put(S.tile + (w / 2) * (NTW * 256));
  }
  if (LG && t < D) {
    double s = 0.0;
#pragma unroll
    for (int i = 0; i < 4; ++i) s += S.part[i][t];
    S.g[t] = s - S.q[t] / prior_var;
  }
  __syncthreads();
  if constexpr (C::H == 1) {
    if (w == 0) {
      add(S.tile);
      // G takes the space of the tiles: every lane's reads before any lane's stores
      // (the LDS accesses of one wave complete in order; this keeps the compiler to it)
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      store(std::integral_constant<int, 0>{});
    }
  } else {
    if (!(w & 1)) add(S.tile + (w / 2) * (NTW * 256));
    __syncthreads();  // both groups have read their tiles before G takes the space
    if (w == 0) store(std::integral_constant<int, 0>{});
    if (w == 2) store(std::integral_constant<int, NTW>{});
  }
  if (VEC && want_gv) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const double s = rows_sum(gvacc[b]);
      if (l < 16) S.part[w][16 * b + l] = s;
    }
  }
  if (LG) loglik = block_sum(S, ll);
  __syncthreads();
  if (VEC && want_gv) {
    if (t < D) {
      double s = 0.0;
#pragma unroll
      for (int i = 0; i < 4; ++i) s += S.part[i][t];
      S.gv[t] = s + vec[t] / prior_var;
    }
    __syncthreads();
  }
}

// want_lg and vec exclude each other.
template <class C>
__device__ __forceinline__ void pass_gram(Smem<C>& S, const double* X, const double* y, int N, int D, double prior_var,
                                          const double* vec, double coef, bool want_lg, bool want_gv, double& loglik) {
  auto run = [&](auto nbc) __attribute__((always_inline)) {
    constexpr int NB = decltype(nbc)::value;
    if (vec != nullptr)
      gram_pass_nb<C, NB, true, false>(S, X, y, N, D, prior_var, vec, coef, want_gv, loglik);
    else if (want_lg)
      gram_pass_nb<C, NB, false, true>(S, X, y, N, D, prior_var, nullptr, 0.0, false, loglik);
    else
      gram_pass_nb<C, NB, false, false>(S, X, y, N, D, prior_var, nullptr, 0.0, false, loglik);
  };
  by_width<C::MAXD>(D, run);
}

template <class C>
__device__ __forceinline__ void pass1(Smem<C>& S, const double* X, const double* y, int N, int D, double prior_var,
                                      bool want_lg, double& loglik) {
  pass_gram(S, X, y, N, D, prior_var, nullptr, 0.0, want_lg, false, loglik);
}

// Load this lane's BS x BS block of S.Gi into registers (entries past D are 0).
template <class C>
__device__ __forceinline__ void load_block(const Smem<C>& S, double (&A)[C::BS][C::BS], int D) {
  const int t = pass_thread();
  const int i0 = C::BS * (t / 16), j0 = C::BS * (t % 16);
#pragma unroll
  for (int a = 0; a < C::BS; ++a)
#pragma unroll
    for (int b = 0; b < C::BS; ++b) {
      const double v = S.Gi[(i0 + a) * C::LDX + j0 + b];
      A[a][b] = (i0 + a < D && j0 + b < D) ? v : 0.0;
    }
}

// Symmetric sweep of the first D pivots: A <- -A^-1, the pivots to S.dk (their
// logarithms belong to pivots_logdet: one log per matrix row instead of one
// in every lane at every pivot).
// Pivots run in groups of BS with the pivot inside a group unrolled, so the
// broadcast row k = BS kk + a is register row a of its owners' blocks.  Every
// lane applies a_ij - a_ik a_kj / d; the owners of the pivot column (a_ik / d),
// the pivot row (a_kj / d) and the pivot (-1/d) then overwrite theirs.
// With zc != nullptr (A positive definite) it also draws pout = chol(A) zc:
// at pivot k the unswept part of row k is the Schur complement's column, so
// L[j][k] = row_k[j] / sqrt(d_k) for j >= k.
template <class C>
__device__ __forceinline__ void sweep(Smem<C>& S, double (&A)[C::BS][C::BS], int D, const double* zc = nullptr,
                                      double* pout = nullptr) {
  constexpr int BS = C::BS;
  const int t = pass_thread();
  const int i0 = BS * (t / 16), j0 = BS * (t % 16);
  double pacc = 0.0;
  for (int kk = 0; kk * BS < D; ++kk) {
    const bool row = t / 16 == kk, col = t % 16 == kk;
#pragma unroll
    for (int a0 = 0; a0 < BS; ++a0) {
      const int k = kk * BS + a0;
      if (k >= D) break;
      double* buf = S.rowbuf[k & 1];
      if (row) {
#pragma unroll
        for (int b = 0; b < BS; ++b) buf[j0 + b] = A[a0][b];
      }
      __syncthreads();
      const double d = buf[k];
      const double rd = 1.0 / d;
      if (t == 0) S.dk[k] = d;
      if (zc != nullptr && t >= k && t < D) pacc = fma(buf[t] * zc[k], 1.0 / sqrt(d), pacc);
      double bjr[BS], sc[BS];
#pragma unroll
      for (int b = 0; b < BS; ++b) bjr[b] = buf[j0 + b] * rd;
#pragma unroll
      for (int a = 0; a < BS; ++a) {
        sc[a] = A[a][a0] * rd;
        const double aik = buf[i0 + a];
#pragma unroll
        for (int b = 0; b < BS; ++b) A[a][b] = fma(-aik, bjr[b], A[a][b]);
      }
#pragma unroll
      for (int a = 0; a < BS; ++a) A[a][a0] = col ? sc[a] : A[a][a0];
#pragma unroll
      for (int b = 0; b < BS; ++b) A[a0][b] = row ? (b == a0 && col ? -rd : bjr[b]) : A[a0][b];
    }
  }
  if (pout != nullptr && t < C::MAXD) pout[t] = t < D ? pacc : 0.0;
}

// log |det A| from the pivots of the last sweep (G +- (eps/2) Omega~ may be
// indefinite); the same in every lane.
template <class C>
__device__ __forceinline__ double pivots_logdet(Smem<C>& S, int D) {
  __syncthreads();  // the last pivot's write
  const int t = pass_thread();
  return block_sum(S, t < D ? log(fabs(S.dk[t])) : 0.0);
}

// Write G^-1 = -A into S.Gi.
template <class C>
__device__ __forceinline__ void store_neg_block(Smem<C>& S, const double (&A)[C::BS][C::BS]) {
  const int t = pass_thread();
  const int i0 = C::BS * (t / 16), j0 = C::BS * (t % 16);
#pragma unroll
  for (int a = 0; a < C::BS; ++a)
#pragma unroll
    for (int b = 0; b < C::BS; ++b) S.Gi[(i0 + a) * C::LDX + j0 + b] = -A[a][b];
}

// Right-looking Cholesky of the leading D x D block of S.Gi in place (lower).
// Column k is scaled after the elimination, so each step reads unscaled
// columns: one barrier per pivot.  Returns log det (= 2 sum log L_kk).
template <class C>
__device__ double cholesky(Smem<C>& S, int D) {
  const int t = pass_thread(), w = t / 64, l = t % 64;
  for (int k = 0; k < D; ++k) {
    const double rd = 1.0 / S.Gi[k * C::LDX + k];
    for (int i = k + 1 + w; i < D; i += 4) {
      const double lik = S.Gi[i * C::LDX + k] * rd;
      for (int j = k + 1 + l; j <= i; j += 64) S.Gi[i * C::LDX + j] -= lik * S.Gi[j * C::LDX + k];
    }
    __syncthreads();
  }
  // pivots d_k sit on the diagonal; scale the columns
  if (t < D) S.qs[t] = sqrt(S.Gi[t * C::LDX + t]);
  __syncthreads();
  double logdet = 0.0;
  for (int k = 0; k < D; ++k) logdet += 2.0 * log(S.qs[k]);
  for (int idx = t; idx < D * D; idx += NT) {
    const int i = idx / D, k = idx % D;
    if (i > k) S.Gi[i * C::LDX + k] /= S.qs[k];
    else if (i == k) S.Gi[i * C::LDX + k] = S.qs[k];
  }
  __syncthreads();
  return logdet;
}

// u = G^-1 p with G^-1 in S.Gi (vector p in LDS): TPR lanes per row.
// Entries past D are written as zeros: the passes over X multiply whole padded
// rows by this vector, and 0 times a stale LDS value left by an earlier kernel
// (possibly Inf or NaN) would not be 0.
template <class C>
__device__ __forceinline__ void ginv_times(Smem<C>& S, const double* p, double* out, int D) {
  constexpr int TPR = NT / C::MAXD;
  const int pt = pass_thread(), r = pt / TPR, h = pt % TPR;
  double s = 0.0;
  if (r < D)
    for (int j = h; j < D; j += TPR) s += S.Gi[r * C::LDX + j] * p[j];
  s = group_sum<TPR>(s);
  __syncthreads();  // out may be p
  if (h == 0) out[r] = r < D ? s : 0.0;
  __syncthreads();
}

// Quadratic-form pass with G^-1 in S.Gi, a_n = x_n^T G^-1 x_n:
//   rmhmc = true : S.dH = X^T [ w (a - b^2)/2 - r ] + q / prior_var, b = X S.u
//   rmhmc = false: S.dH = X^T (w a) = grad log det G.
//
// Lane l = 16 g + m holds row n0 + m's features F(s, g) = 8 (s / 2) + 2 g + s % 2
// (s < 4 NB) of a 16-row block: neighbouring pairs, so that a load brings 16 bytes
// a lane (8-byte loads of X[n0 + m][4 s + g] kept the address unit busy for longer
// than the MFMAs: 122 against 103 us a pass, 2 workgroups per CU, 2048 x 64).  K step s
// of V^T = G^-1 X^T sums over F(s, .); its result slot (t, r) of the lane is the
// feature of x register 4 t + r (rows of the G^-1 operand permuted alike).  G^-1 is
// symmetric, so
// a = sum_t x_t . (2 sum_{t' < t} G^-1_tt' x_t' + G^-1_tt x_t) over 16-feature tiles:
// 2 NB (NB + 1) MFMAs a block (40 at D = 64) in place of 4 NB^2 (64).  At
// capacity 64 the operands of G^-1 (2 NB (NB + 1) doubles a lane) stay in registers for
// the whole pass; at 128 they are read from LDS.
struct Pair {
  double v[2];  // 8-byte aligned: a row of odd D starts anywhere
};

template <class C, int NB, bool RMHMC>
__device__ __forceinline__ void quad_pass_nb(Smem<C>& S, const double* X, const double* y, int N, int D,
                                             double prior_var) {
  constexpr int NS = 4 * NB;
  constexpr bool REG = C::MAXD == 64;
  const int t = pass_thread(), l = t % 64, w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64);
  const int g = l / 16, m = l % 16;
  const int nblk = (N + 15) / 16;
  // G^-1[feature of row m of tile tt][F(s, g)], s < 4 (tt + 1), read as the transposed element
  const int rf = quad_feature(m / 4, m % 4);
  double T[REG ? 2 * NB * (NB + 1) : 1];
  if constexpr (REG) {
    int i = 0;
#pragma unroll
    for (int tt = 0; tt < NB; ++tt)
#pragma unroll
      for (int s = 0; s < 4 * (tt + 1); ++s) T[i++] = S.Gi[quad_feature(s, g) * C::LDX + 16 * tt + rf];
  }
  double dacc[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) dacc[s] = 0.0;
  // features past D, all in the last tile, read feature D - 1 and rows past N row
  // N - 1 (in bounds; they meet zeros of G^-1, q and u, or a weight of zero)
  // (byte offsets from a block's first row, as in gram_loop)
  uint32_t lastb[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) lastb[s] = last_tile_bytes(NB, quad_feature(s, g), D);
  const uint32_t rowb = 8u * (uint32_t)(m * D), gb = 16u * (uint32_t)g;
  auto fetch = [&](auto whole, double (&x)[NS], double& yv, int blk) {
    const int n0 = 16 * min(blk, nblk - 1);
    const char* const Xb = reinterpret_cast<const char*>(X + (size_t)n0 * D);
    const uint32_t row = row_bytes(rowb, n0, N, D);
    const Pair* const xr = reinterpret_cast<const Pair*>(Xb + (row + gb));
#pragma unroll
    for (int s = 0; s < NS - 4; s += 2) {
      const Pair p = xr[2 * s];
      x[s] = p.v[0];
      x[s + 1] = p.v[1];
    }
    if (whole) {
#pragma unroll
      for (int s = NS - 4; s < NS; s += 2) {
        const Pair p = xr[2 * s];
        x[s] = p.v[0];
        x[s + 1] = p.v[1];
      }
    } else {
#pragma unroll
      for (int s = 0; s < 4; ++s) x[NS - 4 + s] = *reinterpret_cast<const double*>(Xb + (row + lastb[s]));
    }
    yv = (y + n0)[min(m, N - n0 - 1)];
  };
  auto block = [&](const double (&x)[NS], double yv, int blk) {
    asm volatile("" ::: "memory");  // q and u (at 128 G^-1 too) are read from LDS per block, not held
    double eta = 0.0, b = 0.0;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      eta = fma(x[s], S.q[quad_feature(s, g)], eta);
      if constexpr (RMHMC) b = fma(x[s], S.u[quad_feature(s, g)], b);
    }
    eta = rows_sum(eta);
    if constexpr (RMHMC) b = rows_sum(b);
    double a = 0.0;
    int i = 0;
#pragma unroll
    for (int tt = 0; tt < NB; ++tt) {
      f64x4 v = f64x4{0, 0, 0, 0};
#pragma unroll
      for (int s = 0; s < 4 * (tt + 1); ++s) {
        if (s == 4 * tt && tt > 0) v *= 2.0;
        const double gi = REG ? T[REG ? i : 0] : S.Gi[quad_feature(s, g) * C::LDX + 16 * tt + rf];
        ++i;
        v = __builtin_amdgcn_mfma_f64_16x16x4f64(gi, x[s], v, 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) a = fma(v[r], x[4 * tt + r], a);
    }
    a = rows_sum(a);
    const bool ok = 16 * blk + m < N;
    const double s = sigmoid(eta);
    const double wv = s * (1.0 - s) * (1.0 - 2.0 * s);
    const double hv = RMHMC ? 0.5 * wv * (a - b * b) - (yv - s) : wv * a;
    const double h = ok ? hv : 0.0;
#pragma unroll
    for (int s2 = 0; s2 < NS; ++s2) dacc[s2] = fma(x[s2], h, dacc[s2]);
  };
  // two register sets in turn (loads one block ahead: with one set, refilled at
  // the block's end, a pass took 235 us in place of 122)
  auto loop = [&](auto whole) {
    double x0[NS], x1[NS], y0, y1;
    if (nblk > 0) fetch(whole, x0, y0, w);
    for (int blk = w; blk < nblk; blk += 8) {
      fetch(whole, x1, y1, blk + 4);
      block(x0, y0, blk);
      fetch(whole, x0, y0, blk + 8);
      if (blk + 4 < nblk) block(x1, y1, blk + 4);
    }
  };
  // a loop of its own for whole tiles keeps the body one basic block (110 -> 101 us);
  // at capacity 128 it spills (189 -> 240 us): there the choice stays inside
  if constexpr (!REG)
    loop(D == 16 * NB);
  else if (D == 16 * NB)
    loop(std::true_type{});
  else
    loop(std::false_type{});
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const double v = group_sum<16>(dacc[s]);
    if (m == 0) S.part[w][quad_feature(s, g)] = v;
  }
  __syncthreads();
  if (t < D) {
    double s = 0.0;
#pragma unroll
    for (int i = 0; i < 4; ++i) s += S.part[i][t];
    S.dH[t] = s + (RMHMC ? S.q[t] / prior_var : 0.0);
  }
  __syncthreads();
}

template <class C>
__device__ __forceinline__ void pass_quad(Smem<C>& S, const double* X, const double* y, int N, int D, double prior_var,
                                          bool rmhmc) {
  by_width<C::MAXD>(D, [&](auto nbc) __attribute__((always_inline)) {
    constexpr int NB = decltype(nbc)::value;
    if (rmhmc)
      quad_pass_nb<C, NB, true>(S, X, y, N, D, prior_var);
    else
      quad_pass_nb<C, NB, false>(S, X, y, N, D, prior_var);
  });
}

template <class C>
__device__ __forceinline__ void pass2(Smem<C>& S, const double* X, const double* y, int N, int D, double prior_var) {
  pass_quad(S, X, y, N, D, prior_var, true);
}

}  // namespace logistic
}  // namespace gjx
