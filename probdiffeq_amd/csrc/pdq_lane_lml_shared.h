// The LML and its reverse adjoint with the square-root factors computed once
// for the whole batch (isotropic, ts0, PDQ_SOLVER).
//
// With ts0, the integrated Wiener prior and a constant output scale every
// factor of the fixed-point smoother's forward pass is a function of the grid
// and the prior alone (solver.step, solvers.py:702-733; the QRs never see a
// mean), and the grid is one for all instances.  The lane kernels
// (pdq_lane_lml.h, pdq_lane_adjoint.h) compute them in every lane of every
// instance and tangent, in one serial chain of 9 400 cycles per grid step, and
// the adjoint once more on its way back.  Here
//  1. lml_chain: one wavefront runs the factors' own chain, the prediction's R_Y
//     and the update (2 400 cycles per step; its lanes take 64 steps'
//     preconditioners at once), and leaves each step's factor and gain;
//  2. lml_revert: one lane per step, the backward conditional's gain and factor;
//  3. lml_merge: one lane per observation interval, the fixed-point merges
//     (estimators_and_losses.py:473-591) of its steps;
//  4. lml_means_part: one lane per instance (and tangent group), the means'
//     recursion through those factors, then the reverse scan (whose factors
//     depend on the instance's observation stds); lml_adjoint_kernel: the scan
//     and the adjoint, which recomputes a tile's means from a checkpoint.
// The grid is cut into chunks of whole intervals, and a launch runs the four
// parts on four successive chunks (lml_parts_kernel): the chain, which leaves
// the chip idle, runs beside the lanes' means.
// What the means' pass reads of a step is the same for every lane: a tile of
// steps is staged in LDS by the wavefront, the next tile's loads under way.
// The order of operations is the lane kernels', the roundings are not: against
// 64-bit arithmetic in another order the gradients' error is 3.3e-14 (the lane
// kernels' 3.6e-14; geometric mean of 20 batches, nu = 3, 4, 64 to 2000 steps),
// on single batches more or less than theirs (1024 instances, 2000 steps: 1.03e-13
// and 1.05e-13 by tangents and adjoint, 0.90e-13 and 0.94e-13 there).
//
// An interval's merges are one lane's, in sequence (1.75 us per step), and an
// interval is not cut: on grids with few observations chain, merges and means run
// one after another (nu = 3, 2000 steps, one interval, 1024 instances: value 5.0
// ms, with tangents 5.8; the lane kernels 7.0 and 7.5).  The records take 552 (nu
// = 3) or 808 (nu = 4) bytes per grid step and call, whatever the batch; the lane
// kernels kept a conditional per observation interval and lane.
//
// 1024 instances, nu = 3, 2000 steps, 101 observations: value 7.29 -> 2.51 ms,
// with the gradient by tangents 7.82 -> 2.68 ms (4.46 with the chain, 2.03, before
// the means, 2.27), by the adjoint 18.2 -> 4.05 ms (5.28;
// 4.49 with the tiles' means recomputed by the wavefront that walks back); 300 instances, nu = 4,
// 500 steps: 4.61 -> 1.33 and 10.95 -> 1.69 ms.  The chain and the means' pass are
// bound by one wavefront's instruction issue.
#pragma once

#include "pdq_lane_adjoint.h"
#include "pdq_lane_lml.h"
#include "pdq_wave.h"

namespace pdq {

// Grid steps staged at once, and per checkpoint of the adjoint (whose two tiles
// of means, and two of records, fit the 160 KB of LDS).
template <int N>
constexpr int lml_tile = N == 4 ? 16 : 12;

// What a step's mean recursion needs of the factors (doubles): P, PI, the
// update's gain, the merge's T = tl_self o to_b (behind an identity: to_b), the
// revert's gain G, the running conditional's A before the step, and the time after it.
template <int N>
struct LmlRec {
  static constexpr int P = 0, PI = N, gain = 2 * N, T = 3 * N, G = 4 * N, A = G + N * N, t = A + N * N,
                       size = t + 1;
};

// The shared buffer: the records of the K - 1 steps; per step (and for the
// final state) the factor before it and the backward conditional's; the
// intervals' conditionals without their means.
template <int N>
struct LmlShared {
  static constexpr int tri = N * (N + 1) / 2, fac = 2 * tri;
  static constexpr int cA = 0, cL = N * N, ctl = cL + tri, cto = ctl + N, cond = cto + N;
  size_t oF, oC, size;
  __host__ __device__ LmlShared(int K, int every) {
    oF = (size_t)(K - 1) * LmlRec<N>::size;
    oC = oF + (size_t)K * fac;
    size = oC + (size_t)((K - 1) / every) * cond;
  }
};

// Interval j's conditional: the shared part and a lane's means (stride).
template <int N, int D>
struct LmlCond {
  using SH = LmlShared<N>;
  const double* __restrict__ f;
  const double* mp;
  size_t stride;
  __device__ __forceinline__ double A(int i, int j) const { return f[SH::cA + i * N + j]; }
  __device__ __forceinline__ double L(int i, int j) const { return j <= i ? f[SH::cL + tri(i, j)] : 0.0; }
  __device__ __forceinline__ double tl(int i) const { return f[SH::ctl + i]; }
  __device__ __forceinline__ double to(int i) const { return f[SH::cto + i]; }
  __device__ __forceinline__ double m(int i, int c) const { return mp[(size_t)(i * D + c) * stride]; }
};

// The left columns of the revert block: rows N..2N-1 are dense, rows 0..N-1
// upper triangular.
template <int N>
struct RevertLeftRows {
  static constexpr bool nz(int, int r) { return r >= N; }
};

// One step of the factors' chain: L -> the update's gain and the next L.
template <int N>
__device__ __forceinline__ void lml_chain_step(const pdq_config& cfg, const double* Q, const double* P,
                                               const double* PI, double s, double* L, double* gain) {
  double big[2 * N * N], PL[N * N];
#pragma unroll
  for (int r = 0; r < N; ++r)
#pragma unroll
    for (int col = 0; col < N; ++col) {
      big[r * N + col] = s * lane_iwp_q<N>(Q, col, r);
      double acc = 0.0;
#pragma unroll
      for (int k = 0; k < N; ++k) {
        const double a = lane_iwp_a<N>(col, k);
        if (a != 0.0 && r <= k) acc += a * (fabs(PI[k]) * L[k * N + r]);
      }
      big[(N + r) * N + col] = acc;
    }
  lane_qr<2 * N, N, RevertLeftRows<N>>(big);
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int j = 0; j < N; ++j) PL[i * N + j] = j <= i ? fabs(P[i]) * big[j * N + i] : 0.0;
  double none[N], Xm[N], mo, oL;
  const double b = 0.0;
#pragma unroll
  for (int i = 0; i < N; ++i) none[i] = i == 1 ? 1.0 : 0.0;
  lane_update<N, 1>(cfg, &b, 0.0, none, PL, Xm, L, &mo, oL, gain);
}

// The factors' chain from step b to step e (one wavefront; the factor before a
// later step than the first is where the previous call left it).
template <int N>
__device__ __forceinline__ void lml_chain(const LmlArgs& a, const pdq_config& cfg, int b, int e, double* pre) {
  constexpr int ps = 2 * N + 2;
  using R = LmlRec<N>;
  using SH = LmlShared<N>;
  const SH lay(a.K, a.every);
  double* const rec = a.shared;
  double* const fac = a.shared + lay.oF;
  double L[N * N], Q[N * N], t = b == 0 ? a.times[0] : rec[(size_t)(b - 1) * R::size + R::t];
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int j = 0; j < N; ++j) {
      if (b == 0) L[i * N + j] = i == j ? (cfg.init_std_rows ? cfg.init_std_rows[i] : cfg.init_std) : 0.0;
      else L[i * N + j] = j <= i ? fac[(size_t)b * SH::fac + tri(i, j)] : 0.0;
      Q[i * N + j] = a.Q[i * N + j];
    }
  auto put = [&](int s) {
    if (threadIdx.x == 0) {
#pragma unroll
      for (int i = 0; i < N; ++i)
#pragma unroll
        for (int j = 0; j <= i; ++j) fac[(size_t)s * SH::fac + tri(i, j)] = L[i * N + j];
    }
  };
  for (int c0 = b; c0 < e; c0 += 64) {
    const int s = c0 + threadIdx.x;
    if (s < e) {
      double P[N], PI[N];
      const double h = a.times[s + 1] - a.times[s];
      lane_precon<N>(h, P, PI);
#pragma unroll
      for (int i = 0; i < N; ++i) {
        pre[threadIdx.x * ps + i] = P[i];
        pre[threadIdx.x * ps + N + i] = PI[i];
        rec[(size_t)s * R::size + R::P + i] = P[i];
        rec[(size_t)s * R::size + R::PI + i] = PI[i];
      }
      pre[threadIdx.x * ps + 2 * N] = lane_noise_scale(cfg, h, 1.0);
      pre[threadIdx.x * ps + 2 * N + 1] = h;
    }
    Grp<64>{}.sync();
    const int n = e - c0 < 64 ? e - c0 : 64;
    auto step = [&](int i, const double* now, double* next) {
      double gain[N];
#pragma unroll
      for (int q = 0; q < ps; ++q) next[q] = pre[(i + 1 < n ? i + 1 : i) * ps + q];
      PDQ_PHASE_BOUNDARY();
      put(c0 + i);
      t += now[2 * N + 1];
      lml_chain_step<N>(cfg, Q, now, now + N, now[2 * N], L, gain);
      if (threadIdx.x == 0) {
        double* const r = rec + (size_t)(c0 + i) * R::size;
#pragma unroll
        for (int q = 0; q < N; ++q) r[R::gain + q] = gain[q];
        r[R::t] = t;
      }
    };
    double x[ps], y[ps];
#pragma unroll
    for (int q = 0; q < ps; ++q) x[q] = pre[q];
    for (int i = 0; i < n; i += 2) {
      step(i, x, y);
      if (i + 1 < n) step(i + 1, y, x);
    }
    Grp<64>{}.sync();
  }
  put(e);
}

// Step s's backward conditional from its factor.
template <int N>
__device__ __forceinline__ void lml_revert(const LmlArgs& a, int s) {
  using R = LmlRec<N>;
  using SH = LmlShared<N>;
  const SH lay(a.K, a.every);
  double* const rec = a.shared + (size_t)s * R::size;
  double* const fac = a.shared + lay.oF + (size_t)s * SH::fac;
  double P[N], PI[N], Xm[N], XL[N * N], Ym[N], YL[N * N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    P[i] = rec[R::P + i];
    PI[i] = rec[R::PI + i];
    Xm[i] = 0.0;
#pragma unroll
    for (int j = 0; j < N; ++j) XL[i * N + j] = j <= i ? fac[tri(i, j)] : 0.0;
  }
  LCond<N, 1> bw;
  lane_revert_prior<N, 1>(a.Q, P, PI, lane_noise_scale(a.cfg, a.times[s + 1] - a.times[s], 1.0), Xm, XL, Ym, YL,
                          LCondViewD<N, 1>{&bw});
#pragma unroll
  for (int e = 0; e < N * N; ++e) rec[R::G + e] = bw.v[CondLayout<N, 1>::A + e];
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int j = 0; j <= i; ++j) fac[SH::tri + tri(i, j)] = bw.L(i, j);
}

// Interval j's merges, in the order of its steps.
template <int N>
__device__ __forceinline__ void lml_merge(const LmlArgs& a, int j) {
  using R = LmlRec<N>;
  using SH = LmlShared<N>;
  const SH lay(a.K, a.every);
  LCond<N, 1> self, bw;
#pragma unroll
  for (int e = 0; e < CondLayout<N, 1>::size; ++e) self.v[e] = bw.v[e] = 0.0;
  for (int e0 = 0; e0 < a.every; ++e0) {
    const size_t s = (size_t)j * a.every + e0;
    double* const rec = a.shared + s * R::size;
    const double* const fac = a.shared + lay.oF + s * SH::fac;
#pragma unroll
    for (int i = 0; i < N; ++i) {
#pragma unroll
      for (int k = 0; k < N; ++k) {
        bw.A(i, k) = rec[R::G + i * N + k];
        bw.setL(i, k, k <= i ? fac[SH::tri + tri(i, k)] : 0.0);
      }
      bw.tl(i) = lane_rcp_nz(rec[R::P + i]);
      bw.to(i) = lane_rcp_nz(rec[R::PI + i]);
      bw.m(i, 0) = 0.0;
      rec[R::T + i] = e0 == 0 ? bw.to(i) : self.tl(i) * bw.to(i);
    }
#pragma unroll
    for (int e = 0; e < N * N; ++e) rec[R::A + e] = self.v[CondLayout<N, 1>::A + e];
    LCond<N, 1> res;
    lane_merge<N, 1>(e0 == 0, LCondViewD<N, 1>{&self}, LCondViewD<N, 1>{&bw}, LCondViewD<N, 1>{&res});
    self = res;
  }
  double* const c = a.shared + lay.oC + (size_t)j * SH::cond;
#pragma unroll
  for (int i = 0; i < N; ++i) {
#pragma unroll
    for (int k = 0; k < N; ++k) {
      c[SH::cA + i * N + k] = self.A(i, k);
      if (k <= i) c[SH::cL + tri(i, k)] = self.L(i, k);
    }
    c[SH::ctl + i] = self.tl(i);
    c[SH::cto + i] = self.to(i);
  }
}

// One step of the means: m and the running conditional's noise mean r, from
// the step's record.
template <int N, int D, int TPL>
__device__ __forceinline__ void lml_mean_step(const pdq_config& cfg, const double* prm, int q0, const double* rec,
                                              const double* A, bool ident, double* m, double* r) {
  constexpr int MC = D * (1 + TPL);
  using R = LmlRec<N>;
  double tmp[N * MC], Pm[N * MC], b[MC], mv[N * MC];
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int c = 0; c < MC; ++c) {
      double acc = 0.0;
#pragma unroll
      for (int k = 0; k < N; ++k) {
        const double av = lane_iwp_a<N>(i, k);
        if (av != 0.0) acc += av * (rec[R::PI + k] * m[k * MC + c]);
      }
      tmp[i * MC + c] = acc + 0.0;
      // rounded here: the value alone and the value with a gradient fuse alike
      Pm[i * MC + c] = wave_rounded(rec[R::P + i] * tmp[i * MC + c]);
    }
  lane_lml_linearize<N, D, TPL>(cfg, prm, q0, Pm, rec[R::t], b);
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int c = 0; c < MC; ++c) {
      double acc = 0.0;
#pragma unroll
      for (int k = 0; k < N; ++k) acc += rec[R::G + i * N + k] * tmp[k * MC + c];
      mv[i * MC + c] = rec[R::T + i] * fma(rec[R::PI + i], m[i * MC + c], -acc);
    }
  if (ident) {
#pragma unroll
    for (int e = 0; e < N * MC; ++e) r[e] = mv[e];
  } else {
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
      for (int c = 0; c < MC; ++c) {
        double acc = 0.0;
#pragma unroll
        for (int k = 0; k < N; ++k) acc += A[i * N + k] * mv[k * MC + c];
        r[i * MC + c] = acc + r[i * MC + c];
      }
  }
#pragma unroll
  for (int c = 0; c < MC; ++c) {
    const double mo = Pm[1 * MC + c] + b[c];
#pragma unroll
    for (int i = 0; i < N; ++i) m[i * MC + c] = Pm[i * MC + c] - rec[R::gain + i] * mo;
  }
}

// A step's record in registers, read a step ahead of its use (without A: read
// where it is used, where the registers do not hold it).
template <int N, bool WITH_A = true>
struct LmlRegs {
  double v[LmlRec<N>::size];
  __device__ __forceinline__ void load(const double* rec) {
#pragma unroll
    for (int e = 0; e < LmlRec<N>::size; ++e)
      if (WITH_A || e < LmlRec<N>::A || e >= LmlRec<N>::t) v[e] = rec[e];
  }
};

// A vector field's parameters in registers (no field of two components reads
// more than four).
struct LmlParams {
  double v[8];
  __device__ __forceinline__ LmlParams(const double* p, int n) {
#pragma unroll
    for (int q = 0; q < 8; ++q) v[q] = q < n ? p[q] : 0.0;
  }
};

// A tile of records on its way to LDS.
template <int N>
struct LmlStage {
  static constexpr int n = lml_tile<N> * LmlRec<N>::size, per = (n + 63) / 64;
  double v[per];
  // the records of steps s0 .. end - 1, at most a tile
  __device__ __forceinline__ void load(const double* __restrict__ shared, int s0, int end) {
    const int count = (end - s0 < lml_tile<N> ? end - s0 : lml_tile<N>) * LmlRec<N>::size;
#pragma unroll
    for (int q = 0; q < per; ++q) {
      const int e = q * 64 + (int)(threadIdx.x & 63);
      if (e < count) v[q] = shared[(size_t)s0 * LmlRec<N>::size + e];
    }
  }
  __device__ __forceinline__ void store(double* lds) const {
#pragma unroll
    for (int q = 0; q < per; ++q) {
      const int e = q * 64 + (int)(threadIdx.x & 63);
      if (e < n) lds[e] = v[q];
    }
  }
};

// The means' pass of a lane from step b (an interval's first) to step e: m and
// the running conditional's noise mean r; `at_step(s, m)` before every step s,
// `at_node(j, r)` with interval j's noise mean after its last step.
template <int N, int D, int TPL, class S, class F>
__device__ __forceinline__ void lml_means_pass(const LmlArgs& a, const pdq_config& cfg, const double* prm, int q0, int b,
                                               int e, double* lds, double* m, double* r, S&& at_step, F&& at_node) {
  const int every = a.every;
  int in = 0, j = b / every;  // the step's place in its interval; the interval
  LmlStage<N> st;
  st.load(a.shared, b, e);
  for (int s0 = b; s0 < e; s0 += lml_tile<N>) {
    Grp<64>{}.sync();
    st.store(lds);
    Grp<64>{}.sync();
    if (s0 + lml_tile<N> < e) st.load(a.shared, s0 + lml_tile<N>, e);
    const int n = e - s0 < lml_tile<N> ? e - s0 : lml_tile<N>;
    constexpr bool with_a = !(N == 5 && TPL == 1);  // (two records with it and four columns: 172 bytes of scratch)
    using Regs = LmlRegs<N, with_a>;
    auto step = [&](int i, const Regs& now, Regs& next) {
      next.load(lds + (i + 1 < n ? i + 1 : i) * LmlRec<N>::size);
      PDQ_PHASE_BOUNDARY();
      at_step(s0 + i, m);
      lml_mean_step<N, D, TPL>(cfg, prm, q0, now.v,
                               with_a ? now.v + LmlRec<N>::A : lds + i * LmlRec<N>::size + LmlRec<N>::A, in == 0, m, r);
      if (++in == every) {
        at_node(j, r);
        in = 0;
        ++j;
      }
    };
    Regs ra, rb;
    ra.load(lds);
    for (int i = 0; i < n; i += 2) {
      step(i, ra, rb);
      if (i + 1 < n) step(i + 1, rb, ra);
    }
  }
}

// The arguments with what an instantiation knows: the vector field is one of
// them, so that a step does not choose among the fields for every component.
__device__ __forceinline__ LmlArgs lml_shared_args(const LmlArgs& args, int field) {
  LmlArgs a = args;
  a.cfg.strategy = PDQ_FIXEDPOINT;
  a.cfg.solver = PDQ_SOLVER;
  a.cfg.constraint = PDQ_TS0;
  a.cfg.re_linearize_after_calibration = 0;
  a.cfg.vector_field = field;
  return a;
}


// The adjoint's storage per lane (doubles): interval means, node data,
// adjoints of the interval means, checkpoints of the mean.
template <int N, int D>
struct LmlAdjShared {
  static constexpr int node = N + 1 + D;
  size_t means, nodes, xibar, ckpt, state, size;
  __host__ __device__ LmlAdjShared(int K, int every) {
    const size_t kobs = (size_t)(K - 1) / every + 1;
    means = 0;
    nodes = means + (kobs - 1) * N * D;
    xibar = nodes + kobs * node;
    ckpt = xibar + (kobs - 1) * N * D;
    state = ckpt + ((size_t)(K - 2) / lml_tile<N> + 1) * N * D;  // m and r between two launches
    size = state + 2 * N * D;
  }
};

// The doubles of the shared buffer and of the lanes' scratch.
inline size_t lml_shared_size(int N, int K, int every) {
  return N == 4 ? LmlShared<4>(K, every).size : LmlShared<5>(K, every).size;
}

inline size_t lml_shared_scratch_size(int N, int D, int tpl, int K, int every, int n_inst, int G, bool reverse) {
  if (reverse) {
    const size_t lanes = (size_t)((n_inst + 63) / 64) * 64;
    return (N == 4 ? LmlAdjShared<4, 2>(K, every).size : LmlAdjShared<5, 2>(K, every).size) * lanes;
  }
  // an interval's noise mean per interval; m and r between two launches
  return ((size_t)((K - 1) / every) + 2) * N * D * (1 + tpl) * n_inst * G;
}

// What one launch does, each part on blocks of its own: the chain of steps
// c0 .. c1, the reverts of steps r0 .. r1, the merges of intervals j0 .. j1 and
// the means' pass of steps m0 .. m1.  A launch's parts work on four successive
// chunks of the grid, so that the chain, one wavefront, runs beside the lanes'
// means; what a part reads was written by earlier launches.
struct LmlParts {
  int c0, c1, r0, r1, j0, j1, m0, m1;
  __host__ __device__ int reverts() const { return (r1 - r0 + 63) / 64; }
  __host__ __device__ int merges() const { return (j1 - j0 + 63) / 64; }
};

// The launches of `steps` grid steps with `lanes` workgroups of means, until one
// fails (not 0).  Up to 64 steps: factors() for all of them (lml_factors_kernel),
// then the means; what such a call costs is its launches.  Beyond, run(parts,
// workgroups) in chunks of whole intervals: launch i runs the chain of chunk i, the reverts of the one before,
// its predecessor's merges and the means of the one before that.  The first three
// launches run without means (24 chunks: an eighth of the chain's time); a chunk
// of fewer than 64 steps (70 us) would not cover its launch, and with fewer than
// six the three launches that fill and drain take what the overlap gives (nu = 4,
// 200 steps, gradient: 0.83 ms in four chunks, 0.77 in one).
template <class F0, class F>
int lml_for_launches(int steps, int every, int lanes, F0&& factors, F&& run) {
  if (steps <= 64) {
    const int rc = factors();
    return rc ? rc : run(LmlParts{0, 0, 0, 0, 0, 0, 0, steps}, 1 + lanes);
  }
  const int target = (steps + 23) / 24 > 64 ? (steps + 23) / 24 : 64;
  const long whole = ((long)target + every - 1) / every * every;
  int chunk = whole < steps ? (int)whole : steps;
  if ((steps + chunk - 1) / chunk < 6) chunk = steps;
  const int n = (steps + chunk - 1) / chunk;
  auto from = [&](int i) { return i < 0 || i >= n ? 0 : i * chunk; };
  auto to = [&](int i) { return i < 0 || i >= n ? 0 : (steps - from(i) < chunk ? steps : from(i) + chunk); };
  for (int i = 0; i < n + 3; ++i) {
    const LmlParts w{from(i),     to(i),     from(i - 1), to(i - 1), from(i - 2) / every, to(i - 2) / every,
                     from(i - 3), to(i - 3)};
    const int rc = run(w, 1 + w.reverts() + w.merges() + (w.m0 < w.m1 ? lanes : 0));
    if (rc) return rc;
  }
  return 0;
}

// The means' pass of a lane per (instance, tangent group) and, after the last
// step, the reverse scan and the outputs.  A lane beyond the last one computes
// it again and writes nothing.
template <int N, int D, int TPL>
__device__ __forceinline__ void lml_means_part(const LmlArgs& a, const LmlParts& w, int block, double* lds) {
  constexpr int MC = D * (1 + TPL);
  using SH = LmlShared<N>;
  const size_t n_lanes = (size_t)a.n_inst * a.G, gl = (size_t)block * 64 + threadIdx.x;
  const bool active = gl < n_lanes;
  const size_t lane = active ? gl : n_lanes - 1;
  const int inst = (int)(lane / a.G), g = (int)(lane % a.G), q0 = g * TPL, ntan = a.n_tan;
  const LmlParams params(a.params + (size_t)inst * a.cfg.n_params, a.cfg.n_params);
  const double* const prm = params.v;
  const double* const tc = a.tcoeffs + (size_t)inst * N * D * (1 + ntan);
  double* const state = a.scratch + (size_t)((a.K - 1) / a.every) * N * MC * n_lanes + lane;
  double m[N * MC], r[N * MC];
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int c = 0; c < MC; ++c) {
      const int tt = c / D - 1, k = c % D, e = i * MC + c;
      if (w.m0 == 0) m[e] = tc[(i * D + k) * (1 + ntan) + (tt < 0 ? 0 : 1 + q0 + tt)];
      else m[e] = state[(size_t)e * n_lanes];
      r[e] = w.m0 == 0 ? 0.0 : state[(size_t)(N * MC + e) * n_lanes];
    }
  lml_means_pass<N, D, TPL>(
      a, a.cfg, prm, q0, w.m0, w.m1, lds, m, r, [](int, const double*) {},
      [&](int j, const double* x) {
        if (active)
#pragma unroll
          for (int e = 0; e < N * MC; ++e) a.scratch[((size_t)j * N * MC + e) * n_lanes + lane] = x[e];
      });
  if (!active) return;
  if (w.m1 < a.K - 1) {
#pragma unroll
    for (int e = 0; e < N * MC; ++e) {
      state[(size_t)e * n_lanes] = m[e];
      state[(size_t)(N * MC + e) * n_lanes] = r[e];
    }
    return;
  }
  const SH lay(a.K, a.every);
  double XL[N * N];
  const double* const fin = a.shared + lay.oF + (size_t)(a.K - 1) * SH::fac;
#pragma unroll
  for (int e = 0; e < N * N; ++e) XL[e] = e % N <= e / N ? fin[tri(e / N, e % N)] : 0.0;
  lane_lml_scan<N, D, TPL>(a, inst, g, m, XL, [&](int j) {
    return LmlCond<N, MC>{a.shared + lay.oC + (size_t)j * SH::cond, a.scratch + (size_t)j * N * MC * n_lanes + lane,
                          n_lanes};
  });
}

// The adjoint's: a lane per instance, with a checkpoint per tile; the mean
// after the last step is left in the state.
template <int N, int D>
__device__ __forceinline__ void lml_means_part_adjoint(const LmlArgs& a, const LmlParts& w, int block, int blocks,
                                                       double* lds) {
  constexpr int ND = N * D;
  const size_t n_lanes = (size_t)blocks * 64, lane = (size_t)block * 64 + threadIdx.x;
  const int inst = lane < (size_t)a.n_inst ? (int)lane : a.n_inst - 1;
  const LmlParams params(a.params + (size_t)inst * a.cfg.n_params, a.cfg.n_params);
  const double* const tc = a.tcoeffs + (size_t)inst * ND * (1 + a.n_tan);
  const LmlAdjShared<N, D> own(a.K, a.every);
  auto at = [&](size_t off) -> double* { return a.scratch + off * n_lanes + lane; };
  double* const state = at(own.state);
  double m[ND], r[ND];
#pragma unroll
  for (int e = 0; e < ND; ++e) {
    m[e] = w.m0 == 0 ? tc[e * (1 + a.n_tan)] : state[(size_t)e * n_lanes];
    r[e] = w.m0 == 0 ? 0.0 : state[(size_t)(ND + e) * n_lanes];
  }
  lml_means_pass<N, D, 0>(
      a, a.cfg, params.v, 0, w.m0, w.m1, lds, m, r,
      [&](int s, const double* x) {
        if (s % lml_tile<N> == 0) {
          double* const c = at(own.ckpt + (size_t)(s / lml_tile<N>) * ND);
#pragma unroll
          for (int e = 0; e < ND; ++e) c[(size_t)e * n_lanes] = x[e];
        }
      },
      [&](int j, const double* x) {
        double* const c = at(own.means + (size_t)j * ND);
#pragma unroll
        for (int e = 0; e < ND; ++e) c[(size_t)e * n_lanes] = x[e];
      });
#pragma unroll
  for (int e = 0; e < ND; ++e) {
    state[(size_t)e * n_lanes] = m[e];
    state[(size_t)(ND + e) * n_lanes] = r[e];
  }
}

// All factors of at most 64 steps by one wavefront: the chain, then a step, then
// an interval, per lane (the barriers: a lane's stores are other lanes' loads).
template <int N>
__global__ void __launch_bounds__(64) lml_factors_kernel(LmlArgs args) {
  __shared__ double lds[64 * (2 * N + 2)];
  const LmlArgs a = lml_shared_args(args, args.cfg.vector_field);
  const int steps = a.K - 1, i = threadIdx.x;
  lml_chain<N>(a, a.cfg, 0, steps, lds);
  __syncthreads();
  if (i < steps) lml_revert<N>(a, i);
  __syncthreads();
  if (i < steps / a.every) lml_merge<N>(a, i);
}

template <int N, int D, int TPL, int FIELD, bool ADJOINT>
__global__ void __launch_bounds__(64) lml_parts_kernel(LmlArgs args, LmlParts w) {
  constexpr int lp = 64 * (2 * N + 2), ls = LmlStage<N>::n;
  __shared__ double lds[lp > ls ? lp : ls];
  const LmlArgs a = lml_shared_args(args, FIELD);
  int b = blockIdx.x;
  if (b == 0) {
    if (w.c0 < w.c1) lml_chain<N>(a, a.cfg, w.c0, w.c1, lds);
    return;
  }
  b -= 1;
  if (b < w.reverts()) {
    const int s = w.r0 + b * 64 + (int)threadIdx.x;
    if (s < w.r1) lml_revert<N>(a, s);
    return;
  }
  b -= w.reverts();
  if (b < w.merges()) {
    const int j = w.j0 + b * 64 + (int)threadIdx.x;
    if (j < w.j1) lml_merge<N>(a, j);
    return;
  }
  b -= w.merges();
  if constexpr (ADJOINT) lml_means_part_adjoint<N, D>(a, w, b, (int)gridDim.x - 1 - w.reverts() - w.merges(), lds);
  else lml_means_part<N, D, TPL>(a, w, b, lds);
}

// A lane per instance, after the means' pass, in two wavefronts: 0 runs the
// reverse scan, its adjoint and the steps' adjoints from the last to the first;
// 1 recomputes the tiles' means from their checkpoints into the lane's column
// of LDS, one tile ahead (beside the scan: the last one).  Both pass one
// barrier per tile.
template <int N, int D, int FIELD>
__global__ void __launch_bounds__(128) lml_adjoint_kernel(LmlArgs args) {
  using R = LmlRec<N>;
  using SH = LmlShared<N>;
  constexpr int ND = N * D, tile = lml_tile<N>;
  __shared__ double stage[2][LmlStage<N>::n];  // one per wavefront
  __shared__ double means[2][tile * ND * 64];
  const int l = threadIdx.x & 63, role = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  double* const lds = stage[role];
  const LmlArgs a = lml_shared_args(args, FIELD);
  const int K = a.K, every = a.every, ntan = a.n_tan;
  const size_t n_lanes = (size_t)gridDim.x * 64, lane = (size_t)blockIdx.x * 64 + l;
  const bool active = lane < (size_t)a.n_inst;
  const int inst = active ? (int)lane : a.n_inst - 1;
  const LmlParams params(a.params + (size_t)inst * a.cfg.n_params, a.cfg.n_params);
  const double* const prm = params.v;
  const double* const tc = a.tcoeffs + (size_t)inst * ND * (1 + ntan);
  const SH lay(K, every);
  const LmlAdjShared<N, D> own(K, every);
  auto at = [&](size_t off) -> double* { return a.scratch + off * n_lanes + lane; };
  const int last = (K - 2) / tile * tile;
  LmlStage<N> st;
  LmlRegs<N> ra, rb;
  auto steps = [&](int s0) { return K - 1 - s0 < tile ? K - 1 - s0 : tile; };
  if (role == 1) {
    if (!a.grad) return;
    double m[ND], r[ND], ck[ND];
    auto fetch = [&](int s0) {
      st.load(a.shared, s0, K - 1);
      const double* const c = at(own.ckpt + (size_t)(s0 / tile) * ND);
#pragma unroll
      for (int e = 0; e < ND; ++e) ck[e] = c[(size_t)e * n_lanes];
    };
    fetch(last);
    for (int s0 = last; s0 >= 0; s0 -= tile) {
      Grp<64>{}.sync();
      st.store(lds);
      Grp<64>{}.sync();
#pragma unroll
      for (int e = 0; e < ND; ++e) {
        m[e] = ck[e];
        r[e] = 0.0;
      }
      if (s0 > 0) fetch(s0 - tile);
      const int n = steps(s0);
      double* const mine = means[s0 / tile & 1] + l;
      auto again = [&](int i, const LmlRegs<N>& now, LmlRegs<N>& next) {
        next.load(lds + (i + 1 < n ? i + 1 : i) * R::size);
        PDQ_PHASE_BOUNDARY();
#pragma unroll
        for (int e = 0; e < ND; ++e) mine[(i * ND + e) * 64] = m[e];
        lml_mean_step<N, D, 0>(a.cfg, prm, 0, now.v, now.v + R::A, true, m, r);  // (r is not used)
      };
      ra.load(lds);
      for (int i = 0; i < n; i += 2) {  // (the last step's result is not used)
        again(i, ra, rb);
        if (i + 1 < n) again(i + 1, rb, ra);
      }
      __syncthreads();  // tile s0 is there, and the walk through the one after it has ended
    }
    return;
  }
  double m[ND];
#pragma unroll
  for (int e = 0; e < ND; ++e) m[e] = at(own.state)[(size_t)e * n_lanes];
  double XL[N * N];
  const double* const fin = a.shared + lay.oF + (size_t)(K - 1) * SH::fac;
#pragma unroll
  for (int e = 0; e < N * N; ++e) XL[e] = e % N <= e / N ? fin[tri(e / N, e % N)] : 0.0;
  auto cond = [&](int j) {
    return LmlCond<N, D>{a.shared + lay.oC + (size_t)j * SH::cond, at(own.means + (size_t)j * ND), n_lanes};
  };
  auto node = [&](int j) { return at(own.nodes + (size_t)j * LmlAdjShared<N, D>::node); };
  const double lp = adj_scan<N, D>(a, inst, m, XL, n_lanes, cond, node);
  if (a.value && active) a.value[inst] = lp;
  if (!a.grad) return;
  double mbar[ND], cbar[ND], tbar[8];
  adj_scan_adjoint<N, D>(a, n_lanes, cond, node, [&](int j) { return at(own.xibar + (size_t)j * ND); }, mbar);
  // (every divides the grid's steps: the terminal marginal stands behind an identity)
#pragma unroll
  for (int e = 0; e < ND; ++e) cbar[e] = 0.0;
#pragma unroll
  for (int q = 0; q < 8; ++q) tbar[q] = 0.0;
  const int np = a.cfg.n_params < 8 ? a.cfg.n_params : 8;
  struct Self {
    const double* rec;
    __device__ double tl(int) const { return 1.0; }  // (T holds both scales)
    __device__ double A(int i, int k) const { return rec[R::A + i * N + k]; }
  };
  st.load(a.shared, last, K - 1);
  int in = 0, j = (K - 1) / every;  // the place of the step after the current one in its interval, that interval
  for (int s0 = last; s0 >= 0; s0 -= tile) {
    Grp<64>{}.sync();
    st.store(lds);
    Grp<64>{}.sync();
    if (s0 > 0) st.load(a.shared, s0 - tile, K - 1);
    const int n = steps(s0);
    const double* const mine = means[s0 / tile & 1] + l;
    __syncthreads();
    auto back = [&](int i, const LmlRegs<N>& now, LmlRegs<N>& next) {
      const double* const rec = now.v;
      next.load(lds + (i > 0 ? i - 1 : 0) * R::size);
      PDQ_PHASE_BOUNDARY();
      if (in == 0) {
        // after this step a reset stored the running conditional as interval
        // j - 1's: its adjoint comes from the scan
        --j;
        in = every;
        const double* const xb = at(own.xibar + (size_t)j * ND);
#pragma unroll
        for (int e = 0; e < ND; ++e) cbar[e] = xb[(size_t)e * n_lanes];
      }
      --in;
      double Pm[D];
#pragma unroll
      for (int c = 0; c < D; ++c) {
        double acc = 0.0;
#pragma unroll
        for (int k = 0; k < N; ++k) acc += lane_iwp_a<N>(0, k) * (rec[R::PI + k] * mine[(i * ND + k * D + c) * 64]);
        Pm[c] = rec[R::P] * (acc + 0.0);
      }
      adj_back_step<N, D>(a.cfg, prm, np, rec + R::P, rec + R::PI, rec + R::G, rec + R::T, rec + R::gain, Pm, in == 0,
                          Self{rec}, mbar, cbar, tbar);
    };
    ra.load(lds + (n - 1) * R::size);
    for (int i = n - 1; i >= 0; i -= 2) {
      back(i, ra, rb);
      if (i > 0) back(i - 1, rb, ra);
    }
  }
  for (int q = 0; q < ntan; ++q) {
    double g = 0.0;
#pragma unroll
    for (int e = 0; e < 8; ++e) g = e == q && q < np ? tbar[e] : g;
#pragma unroll
    for (int e = 0; e < ND; ++e) g += mbar[e] * tc[(size_t)e * (1 + ntan) + 1 + q];
    if (active) a.grad[(size_t)inst * ntan + q] = g;
  }
}

}  // namespace pdq
