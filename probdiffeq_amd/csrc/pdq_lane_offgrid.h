// Off-grid marginals of a solution (ProbabilisticSolver.offgrid_marginals,
// solvers.py:149-203), isotropic, one lane per query time.
//
// For a query t the lane finds the grid interval (t0, t1] by
// searchsorted(t_grid, t) (side "left", as the reference) and evaluates
// * the filter (estimators_and_losses.py:403-414): the marginal at t0
//   predicted to t with the transition of t1's output scale;
// * the fixed-interval smoother (:674-707): the filtering marginal at t0
//   reverted to t and on to t1; the smoothed marginal at t1 marginalised
//   back through the conditional t1 -> t.
// The per-query algebra is the lane solve's (pdq_lane.h), all in registers.
// Like the reference, t must lie strictly inside the grid and off its
// points; other t give an unspecified result (the interval index is clamped
// to [1, K - 1], so every access stays inside the solution arrays).
#pragma once

#include "pdq_lane.h"
#include "pdq_wave.h"

namespace pdq {

// The grid interval (ts[i - 1], ts[i]] of t.
__device__ __forceinline__ int lane_offgrid_interval(const double* ts, int K, double t) {
  int lo = 0, hi = K;
  while (lo < hi) {  // first index with ts[i] >= t: at most log2(K) + 1 rounds
    const int mid = (lo + hi) / 2;
    if (ts[mid] < t) lo = mid + 1;
    else hi = mid;
  }
  return lo < 1 ? 1 : (lo > K - 1 ? K - 1 : lo);
}

// The marginal at t in (t0, t1] from the rows of t0, (m0, L0), and (smoother)
// of t1, (m1, L1), which load1() fetches when they are needed.
template <int N, int D, int STRATEGY, class F>
__device__ __forceinline__ void lane_offgrid_marginal(const OffgridArgs& a, double t, double t0, double t1, double os,
                                                      const double* m0, const double* L0, F&& load1, double* Ym,
                                                      double* YL) {
  const pdq_config& cfg = a.cfg;
  double P[N], PI[N];
  lane_precon<N>(t - t0, P, PI);
  const double s0 = lane_noise_scale(cfg, t - t0, os);
  if constexpr (STRATEGY == PDQ_FILTER) {
    lane_marginalise_prior<N, D>(a.Q, P, PI, s0, m0, L0, Ym, YL);
  } else {
    double Xm[N * D], XL[N * N], Zm[N * D], ZL[N * N], m1[N * D], L1[N * N];
    LCond<N, D> c_t_t0, c_t1_t;
    lane_revert_prior<N, D>(a.Q, P, PI, s0, m0, L0, Xm, XL, c_t_t0);
    lane_precon<N>(t1 - t, P, PI);
    const double s1 = lane_noise_scale(cfg, t1 - t, os);
    lane_revert_prior<N, D>(a.Q, P, PI, s1, Xm, XL, Zm, ZL, c_t1_t);
    load1(m1, L1);
    lane_marginalise_cond<N, D>(c_t1_t, m1, L1, Ym, YL);
  }
}

// Two neighbouring doubles (8-byte aligned).
struct alignas(8) OffgridPair {
  double v[2];
};
typedef double OffgridVec __attribute__((vector_size(16), aligned(8)));

// One wavefront's 64 queries.  What bounds them beside the smoother's two
// reverts per query (2650 FP64 instructions at nu = 4) is the memory
// interface: a lane's own loads and stores touch a cache line per lane and
// instruction.  So the wavefront gathers the rows of its queries together, 12
// lanes along a 25-entry row, through LDS (an odd number of doubles per
// query: a lane's column falls on banks of its own), both grid points' rows
// before the first of them is used, and writes its results as one piece, with
// stores that leave the L2 to the rows.  The grid is searched in LDS when the
// queries are of one instance.
// 4096 instances x 256 queries on 200 points, nu = 4, smoother: 198 -> 167 us
// with sorted queries (0.78 GB: 4.7 TB/s, a large copy reaches 4.8), 284 -> 228
// with random ones; filter, random: 205 -> 133 us.
template <int N, int D>
struct OffgridTile {
  static constexpr int nn = N * N, nd = N * D, os = nn + nd;
  static constexpr int stride = os | 1;
  static constexpr int lds = 64 * stride;  // doubles
};

// The rows rows[j] + off, j = 0..63, of a matrix of n-double rows: pairs (and
// an odd row's last double) into registers, then into the queries' LDS rows
// at `to`.
template <int n>
struct OffgridGather {
  static constexpr int np = n / 2;
  OffgridPair p[np];
  double last;
  __device__ __forceinline__ void load(const double* __restrict__ src, const size_t* rows, int off, int l) {
#pragma unroll
    for (int q = 0; q < np; ++q) {
      const int e = q * 64 + l;
      p[q] = *reinterpret_cast<const OffgridPair*>(src + ((rows[e / np] + off) * n + 2 * (e % np)));
    }
    if (n % 2) last = src[(rows[l] + off) * n + n - 1];
  }
  __device__ __forceinline__ void store(double* lds, int stride, int to, int l) const {
#pragma unroll
    for (int q = 0; q < np; ++q) {
      const int e = q * 64 + l;
      double* const d = lds + (e / np) * stride + to + 2 * (e % np);
      d[0] = p[q].v[0];
      d[1] = p[q].v[1];
    }
    if (n % 2) lds[l * stride + to + n - 1] = last;
  }
};

// `count` queries' rows of n doubles from LDS to dst (a multiple of 64 queries
// into its array), in pairs.
template <int n>
__device__ __forceinline__ void offgrid_store(double* __restrict__ dst, const double* lds, int stride, int from,
                                              int count, int l) {
#pragma unroll
  for (int q = 0; q < (n + 1) / 2; ++q) {
    const int e = 2 * (q * 64 + l);  // the first of two neighbouring doubles of the piece
    if (e + 1 < count * n)
      __builtin_nontemporal_store(OffgridVec{lds[(e / n) * stride + from + e % n],
                                             lds[((e + 1) / n) * stride + from + (e + 1) % n]},
                                  reinterpret_cast<OffgridVec*>(dst + e));
    else if (e < count * n) dst[e] = lds[(e / n) * stride + from + e % n];
  }
}

template <int N, int D, int STRATEGY>
__device__ __forceinline__ void wave_offgrid(const OffgridArgs& a, size_t q0, int count, double* lds, size_t* rows) {
  using T = OffgridTile<N, D>;
  const int K = a.K, l = threadIdx.x;
  const size_t q = q0 + (l < count ? l : count - 1);  // lanes without a query repeat the last one
  const size_t inst = q / (size_t)a.n_query;
  const double* __restrict__ ts = a.times + inst * K;
  const double t = a.t_query[q];
  int i;
  const size_t first = q0 / (size_t)a.n_query;
  if (K <= T::lds && (q0 + count - 1) / (size_t)a.n_query == first) {
    for (int e = l; e < K; e += 64) lds[e] = a.times[first * K + e];
    Grp<64>{}.sync();
    i = lane_offgrid_interval(lds, K, t);
  } else {
    i = lane_offgrid_interval(ts, K, t);
  }
  const double t0 = ts[i - 1], t1 = ts[i];
  const double os = a.output_scale[inst * K + i];
  rows[l] = inst * K + (i - 1);
  Grp<64>{}.sync();
  double* const own = lds + l * T::stride;
  double m0[T::nd], L0[T::nn], Ym[T::nd], YL[T::nn];
  // the rows of t0 and (smoother) of t1: both on their way before the first is
  // needed, then one after the other through the same LDS
  {
    const int g = wave_here(l);  // (its offsets are not kept beyond the gathers)
    OffgridGather<T::nn> gL, hL;
    OffgridGather<T::nd> gm, hm;
    gL.load(STRATEGY == PDQ_FILTER ? a.chol : a.filt_chol, rows, 0, g);
    gm.load(STRATEGY == PDQ_FILTER ? a.mean : a.filt_mean, rows, 0, g);
    if constexpr (STRATEGY != PDQ_FILTER) {
      hL.load(a.chol, rows, 1, g);
      hm.load(a.mean, rows, 1, g);
    }
    gL.store(lds, T::stride, 0, g);
    gm.store(lds, T::stride, T::nn, g);
    Grp<64>{}.sync();
#pragma unroll
    for (int e = 0; e < T::nn; ++e) L0[e] = own[e];
#pragma unroll
    for (int e = 0; e < T::nd; ++e) m0[e] = own[T::nn + e];
    Grp<64>{}.sync();
    if constexpr (STRATEGY != PDQ_FILTER) {
      hL.store(lds, T::stride, 0, g);
      hm.store(lds, T::stride, T::nn, g);
      Grp<64>{}.sync();
    }
    PDQ_PHASE_BOUNDARY();
  }
  lane_offgrid_marginal<N, D, STRATEGY>(
      a, t, t0, t1, os, m0, L0,
      [&](double* m1, double* L1) {
#pragma unroll
        for (int e = 0; e < T::nn; ++e) L1[e] = own[e];
#pragma unroll
        for (int e = 0; e < T::nd; ++e) m1[e] = own[T::nn + e];
      },
      Ym, YL);
#pragma unroll
  for (int e = 0; e < T::nn; ++e) own[e] = YL[e];
#pragma unroll
  for (int e = 0; e < T::nd; ++e) own[T::nn + e] = Ym[e];
  Grp<64>{}.sync();
  const int s = wave_here(l);
  offgrid_store<T::nn>(a.chol_out + q0 * T::nn, lds, T::stride, 0, count, s);
  offgrid_store<T::nd>(a.mean_out + q0 * T::nd, lds, T::stride, T::nn, count, s);
  Grp<64>{}.sync();
}

template <int N, int D, int STRATEGY>
__global__ void __launch_bounds__(64, 2) lane_offgrid_kernel(OffgridArgs a) {
  __shared__ double lds[OffgridTile<N, D>::lds];
  __shared__ size_t rows[64];
  const size_t total = (size_t)a.n_inst * a.n_query;
  const size_t stride = (size_t)gridDim.x * 64;
  for (size_t q = (size_t)blockIdx.x * 64; q < total; q += stride)
    wave_offgrid<N, D, STRATEGY>(a, q, (int)(total - q < 64 ? total - q : 64), lds, rows);
}

}  // namespace pdq
