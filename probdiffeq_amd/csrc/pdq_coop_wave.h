// The cooperative solver for fixed shapes: one IVP instance per wavefront,
// every matrix size a compile-time constant, the QR in registers (pdq_wave.h).
//
// It computes what the run-time-shape kernel (pdq_coop.hip) computes with 64
// lanes per instance, in the same order of operations, so that for finite
// data every output is the same bit for bit.  What bounds both is the latency
// of one instance's serial chain (a few QRs of 10 to 24 rows per attempt; a
// batch of 1024 has one wavefront per SIMD).  The run-time-shape kernel spends
// that chain on LDS round trips: every operand of every reflector, with
// run-time loop bounds.  Here
// * lane j holds column j of a stack in registers and builds it there from the
//   factors in LDS (lane i then also owns row i of the resulting factor);
// * the zeros of the stacks (triangular factors, the IWP transition kron(A, I),
//   the observation's two derivatives) are skipped at compile time;
// * the loop is a state machine whose operations share one prediction: an
//   attempt and the two halves of an interpolation (as in pdq_lane.h), so that
//   a kernel holds each piece of code once;
// * the solve's scalars (t, dt, output scale, counts) are wave-uniform
//   registers, and every loop and branch on them is a scalar one.
// Measured on one MI355X, the same outputs bit for bit: 1024 dense
// Lotka-Volterra solves (nu = 4, filter, 200 points) 71.3 -> 10.6 ms, one such
// solve 32.3 -> 5.6 ms, 1024 stiff van der Pol solves (nu = 5, ts1) 20.9 -> 3.1 ms.
// Of the 14.3 ms of a first version, 3.7 went with the solve's scalars in
// vector registers under scalar branches (spilled scalar registers before), no
// padding in the structs that are copied (padded copies went through scratch
// memory), the reflectors broadcast by one DPP move per value where the columns
// fit a row of 16 lanes (two v_readlane before), the next point's time loaded a
// point ahead, and the outputs' addresses loaded in one batch.
// Configurations it does not hold (error_state_std, re-linearisation, Monte
// Carlo Jacobians, the LML) stay with the run-time-shape kernel.
#pragma once

#include "pdq_args.h"
#include "pdq_pade.h"
#include "pdq_wave.h"

namespace pdq {

// A fixed shape: N = nu + 1, d, dense or isotropic, smoother or filter, IWP or
// exponential prior.
template <int N_, int D_, bool DENSE_, bool SMOOTHER_, bool EXPO_ = false>
struct WShape {
  static constexpr int N = N_, d = D_;
  static constexpr bool dense = DENSE_, smoother = SMOOTHER_, expo = EXPO_;
  static constexpr int nc = dense ? N * d : N, mc = dense ? 1 : d, ko = dense ? d : 1;
  static constexpr int st = dense && !expo ? d : 1;  // stride of the transition's non-zeros
  static constexpr int nn = nc * nc, ms = nc * mc;
  // LDS (doubles): the transition, then the instance
  static constexpr int oA = 0, oQ = oA + nn;
  static constexpr int oP = oQ + nn, oPI = oP + nc;
  static constexpr int oUm = oPI + nc, oPm = oUm + ms, oPL = oPm + ms, oTmp = oPL + nn;
  // a conditional: A, mean, factor, to_latent, to_observed
  static constexpr int cA = 0, cm = cA + nn, cL = cm + ms, ctl = cL + nn, cto = ctl + nc, csize = cto + nc;
  static constexpr int oB = oTmp + ms, oE = oB + (smoother ? csize : 0);
  // three solution slots: mean, factor, conditional
  static constexpr int sm = 0, sL = sm + ms, sC = sL + nn, ssize = sC + (smoother ? csize : 0);
  static constexpr int oS = oE + (smoother ? csize : 0);
  // the exponential prior's drift rows and the scratch of its transition
  static constexpr int m10 = 10 * d;  // columns of the Legendre terms
  static constexpr int xD = oS + 3 * ssize, xp = xD + (expo ? d * nc : 0), xB = xp + nn, x2 = xB + nc * d, x4 = x2 + nn,
                       x6 = x4 + nn, x8 = x6 + nn, xT = x8 + nn, xV = xT + nn, xW = xV + nn, xPB = xW + nn,
                       xR = xPB + nc * d, xend = xR + nc * m10;
  static constexpr int oPrm = expo ? xend : xD;
  static constexpr int fixed_size = oPrm;  // + n_params
  static_assert(2 * nc <= 32, "a column of the revert block per lane, a power per half wavefront");
  static_assert(N >= 2 && d <= 2, "the observation's rows and the columns' sums");
  static_assert(!expo || (dense && 2 * nc + m10 <= 64), "a column of the linear system per lane");
};

// The stacks' patterns (WaveQrPlan).
template <class SH>
struct WPatStack {  // [dense; upper triangle]
  static constexpr int nc = SH::nc, M = 2 * nc, NP = nc, MROWS = M, COLS = nc;
  static constexpr int row(int r) { return r; }
  static constexpr bool nz(int r, int c) { return r < nc || r - nc <= c; }
};
template <class SH>
struct WPatRevert {  // [[upper triangle, 0], [dense, upper triangle]]
  static constexpr int nc = SH::nc, M = 2 * nc, NP = M, MROWS = M, COLS = M;
  static constexpr int row(int r) { return r; }
  static constexpr bool nz(int r, int c) { return c < nc ? (r >= nc || r <= c) : (r >= nc && r - nc <= c - nc); }
};
template <class SH>
struct WPatUpdate {  // [[diagonal, 0], [(H L)^T, L^T]]: H reads derivatives 0 and 1, the first 2 ko rows of L
  static constexpr int nc = SH::nc, ko = SH::ko, M = ko + nc, NP = M, MROWS = M, COLS = M;
  static constexpr int row(int r) { return r; }
  static constexpr bool nz(int r, int c) { return r < ko ? r == c : (c < ko ? r - ko < 2 * ko : r - ko <= c - ko); }
};
template <class SH>
struct WPatTall {  // the Legendre terms: dense
  static constexpr int nc = SH::nc, M = SH::m10, NP = nc, MROWS = M, COLS = nc;
  static constexpr int row(int r) { return r; }
  static constexpr bool nz(int, int) { return true; }
};
template <class SH>
struct WPatDouble {  // [upper triangle; dense]
  static constexpr int nc = SH::nc, M = 2 * nc, NP = nc, MROWS = M, COLS = nc;
  static constexpr int row(int r) { return r; }
  static constexpr bool nz(int r, int c) { return r >= nc || r <= c; }
};
template <class SH>
struct WPatFx {  // [(H L)^T; diagonal], without (H L)^T's zero rows
  static constexpr int nc = SH::nc, ko = SH::ko, M = 3 * ko, NP = ko, MROWS = nc + ko, COLS = ko;
  static constexpr int row(int r) { return r < 2 * ko ? r : nc + r - 2 * ko; }
  static constexpr bool nz(int r, int c) { return r < 2 * ko || r - 2 * ko == c; }
};

// Orders the wavefront's LDS accesses.
__device__ __forceinline__ void wave_sync() { Grp<64>{}.sync(); }

template <int n>
__device__ __forceinline__ void wave_copy(int l, double* dst, const double* src) {
#pragma unroll
  for (int e0 = 0; e0 < n; e0 += 64) {
    const int e = e0 + l;
    if (e < n) dst[e] = src[e];
  }
}

// A solution's scalars (the same in every lane).  No padding: copies of a
// padded struct go through scratch memory.
struct WScal {
  double t, os, mle_run, mle_n;
  int nsteps, ident;
};

// The linearisation: the operator's non-zero block J (ko x 2 ko, derivatives 0
// and 1; ts1 only) and b (ko x mc), in every lane.
template <class SH>
struct WLin {
  double J[SH::ko * 2 * SH::ko], b[SH::ko * SH::mc];
};

// The step's quantities that its parts hand on (uniform).
struct WErr {
  double oL[4];  // the error model's observed factor (ko x ko)
  double sigma;
};

// The launch's arguments, in the kernel argument segment.  The solve reads them
// through a pointer that it renews in every iteration (WCtx::renew): what an
// iteration needs is then loaded in it (scalar loads, cached) instead of ahead
// of the loop, where it would take scalar registers throughout and be spilled.
#ifdef PDQ_HOST_EMU
using WArgs = const KArgs;
#else
using WArgs = const __attribute__((address_space(4))) KArgs;
#endif

// The configuration an attempt reads, in scalar registers for the whole solve.
struct WCfg {
  double rtol, atol, eps, damp, safety, factor_min, factor_max;
  int ts1, vector_field, error_norm, integral, clip_dt, max_attempts;
  template <class Cfg>
  __device__ __forceinline__ explicit WCfg(const Cfg& c)
      : rtol(c.rtol), atol(c.atol), eps(c.eps), damp(c.damp), safety(c.safety), factor_min(c.factor_min),
        factor_max(c.factor_max), ts1(c.constraint == PDQ_TS1), vector_field(c.vector_field),
        error_norm(c.error_norm), integral(c.control == PDQ_CONTROL_INTEGRAL), clip_dt(c.clip_dt),
        max_attempts(c.max_attempts) {}
};

// The exponential prior's constants of a lane: rhs lane 2 nc + q of the linear
// system holds column q of the Legendre terms (block q / d), with the block's
// coefficients and the root of 2 block + 1.
struct WLegendre {
  double c[5], den, rden;
  __device__ __forceinline__ WLegendre(int col, int d) {
    int blk = col < 0 ? 0 : col / d;
    blk = blk < 10 ? blk : 9;
#pragma unroll
    for (int kk = 0; kk < 5; ++kk) {
      // row `blk` of the table by selection: the index differs between lanes
      double v = 0.0;
#pragma unroll
      for (int b = 0; b < 10; ++b) v = blk == b ? legendre9(b, 2 * kk + (b & 1)) : v;
      c[kk] = v;
    }
    den = sqrt((double)(2 * blk + 1));
    rden = 1.0 / den;
  }
};

template <class SH>
struct WCtx {
  WArgs* a;
  WCfg cfg;
  double* lds;
  int l, inst, K;
  bool dynamic;  // solver_dynamic
  double base_scale;
  WLegendre lg;
  __device__ __forceinline__ double* P() const { return lds + SH::oP; }
  __device__ __forceinline__ double* PI() const { return lds + SH::oPI; }
  __device__ __forceinline__ const double* A() const { return lds + SH::oA; }
  __device__ __forceinline__ const double* Q() const { return lds + SH::oQ; }
  __device__ __forceinline__ const double* prm() const { return lds + SH::oPrm; }
  __device__ __forceinline__ double* slot(int s) const { return lds + SH::oS + s * SH::ssize; }
  __device__ __forceinline__ WCtx(WArgs* args, double* lds_, int lane) : a(args), cfg(args->cfg), lds(lds_), l(lane), inst(0), K(args->K), dynamic(args->cfg.solver == PDQ_SOLVER_DYNAMIC),
        base_scale(args->cfg.base_output_scale), lg(SH::expo ? lane - 2 * SH::nc : 0, SH::d) {}
  __device__ __forceinline__ bool ts1() const { return cfg.ts1 != 0; }
  __device__ __forceinline__ void renew() {
#ifndef PDQ_HOST_EMU
    asm("" : "+s"(a));
#endif
  }
};

// preconditioner_taylor (utilities.py:74-84) into P and PI, and dt^nord (in
// every lane): one evaluation of pow, lanes 0.. the powers, lanes 32.. their
// inverses, lane 31 dt^nord.
template <class SH>
__device__ __forceinline__ double w_precon(const WCtx<SH>& c, double dt, int nord) {
  const int i = c.l & 31, pw = i < SH::nc ? SH::N - 1 - (SH::dense ? i / SH::d : i) : 0;
  const int ex = c.l == 31 ? nord : (c.l < 32 ? pw : -pw);
  const double s = factorial_d(pw), p = pow(dt, (double)ex);
  if (i < SH::nc) (c.l < 32 ? c.P() : c.PI())[i] = c.l < 32 ? p / s : p * s;
  wave_sync();
  return wave_bcast(p, 31);
}

// Row i's lane: lane i < nc (the others repeat row nc - 1 and write nothing).
template <class SH>
__device__ __forceinline__ int w_row(const WCtx<SH>& c) {
  return c.l < SH::nc ? c.l : SH::nc - 1;
}

// Z = X Y for n x n matrices in LDS (Z another one), each product's sum in
// ascending order: a lane takes W consecutive entries of one row.
template <int n>
__device__ __forceinline__ void w_gemm(int l, const double* X, const double* Y, double* Z) {
  constexpr int W = n * n <= 64 ? 1 : (n * n <= 128 ? 2 : 3);
  static_assert(n % W == 0 && n * (n / W) <= 64, "one lane per W entries");
  constexpr int per = n / W, lanes = n * per;
  const int t = l < lanes ? l : lanes - 1, i = t / per, j = (t % per) * W;
  double acc[W] = {};
#pragma unroll
  for (int q = 0; q < n; ++q) {
    const double x = X[i * n + q];
#pragma unroll
    for (int w = 0; w < W; ++w) acc[w] += x * Y[q * n + j + w];
  }
  if (l < lanes)
#pragma unroll
    for (int w = 0; w < W; ++w) Z[i * n + j + w] = acc[w];
  wave_sync();
}

// Z = X B for an n x n matrix X and n x d columns B.
template <int n, int d>
__device__ __forceinline__ void w_gemm_cols(int l, const double* X, const double* B, double* Z) {
  static_assert(n * d <= 64, "a lane per entry");
  const int t = l < n * d ? l : n * d - 1, i = t / d, k = t % d;
  double acc = 0.0;
#pragma unroll
  for (int q = 0; q < n; ++q) acc += X[i * n + q] * B[q * d + k];
  if (l < n * d) Z[t] = acc;
  wave_sync();
}

// DenseExponential.transition (ssm_impl_dense.py:405-423) for the step dt:
// e^{A_p} into A and the lower-triangular Gramian factor U into Q, as
// exp_transition (pdq_coop.hip) forms them: A_p = dt p^-1 A p, B_p = sqrt|dt|
// |p^-1| B, scaling by 2^-s, the degree-9 Pade / Legendre approximation, s
// doublings, non-negative diagonal (exp_gram_cholesky, util/gram_util.py:
// 17-77).  The linear system's columns (the denominator's, the numerator's,
// the Legendre terms') are held one per lane: its LU with partial pivoting
// eliminates all of them at once, and the back substitution runs on the
// right-hand sides' lanes.  Its time is the instructions of one wavefront, a
// few thousand in sequence; the run-time-shape form waited for LDS operands.
// 200 Matern solves (nu = 4, d = 2, 20 points): 154 -> 24.5 ms, the same bits.
template <class SH>
__device__ __forceinline__ void w_exp_transition(const WCtx<SH>& c, double dt) {
  constexpr int n = SH::nc, d = SH::d, N = SH::N, nn = SH::nn, m10 = SH::m10;
  const int l = c.l;
  double* const lds = c.lds;
  double *const eA = lds + SH::oA, *const U = lds + SH::oQ, *const Ap = lds + SH::xp, *const Bp = lds + SH::xB;
  double *const A2 = lds + SH::x2, *const A4 = lds + SH::x4, *const A6 = lds + SH::x6, *const A8 = lds + SH::x8;
  double *const T = lds + SH::xT, *const V = lds + SH::xV, *const W = lds + SH::xW, *const PB = lds + SH::xPB;
  double* const rhs = lds + SH::xR;
  const double base = c.base_scale;
#pragma unroll
  for (int e0 = 0; e0 < nn; e0 += 64) {
    const int e = e0 + l < nn ? e0 + l : nn - 1, i = e / n, j = e % n;
    const double drift = lds[SH::xD + (i < n - d ? j : (i - (n - d)) * n + j)];
    const double a = i < n - d ? (j == i + d ? 1.0 : 0.0) : drift;
    const double v = ((dt * c.PI()[i]) * a) * c.P()[j];
    if (e0 + l < nn) Ap[e] = v;
  }
  if (l < n * d) {
    const int i = l / d, k = l % d;
    Bp[l] = (sqrt(fabs(dt)) * fabs(c.PI()[i])) * (i == (N - 1) * d + k ? base : 0.0);
  }
  wave_sync();
  // _exp_gram_cholesky_init: the number of doublings from the 1-norm
  double a_l1;
  {
    const int j = w_row(c);
    double s = 0.0;
#pragma unroll
    for (int i = 0; i < n; ++i) s += fabs(Ap[i * n + j]);
    s = fmax(0.0, s);
    a_l1 = 0.0;
#pragma unroll
    for (int q = 0; q < n; ++q) a_l1 = fmax(a_l1, wave_bcast(s, q));
  }
  const double s1 = log2(a_l1 / 0.41098379928173995), s2 = log2((double)(n - 1) / 9.0);
  // at most 64 doublings (a 1-norm up to 0.41 2^64): a larger or non-finite
  // norm gives a non-finite transition either way, and the loop stays bounded
  double num = fmax(0.0, ceil(fmax(s1, s2)));
  if (!(num <= 64.0)) num = 64.0;
  const int nd = wave_int((int)num);
  const double two = ldexp(1.0, nd), sq = sqrt(two);
#pragma unroll
  for (int e0 = 0; e0 < nn; e0 += 64)
    if (e0 + l < nn) Ap[e0 + l] = (1.0 / two) * Ap[e0 + l];
  if (l < n * d) Bp[l] = Bp[l] / sq;
  wave_sync();
  w_gemm<n>(l, Ap, Ap, A2);
  w_gemm<n>(l, A2, A2, A4);
  w_gemm<n>(l, A4, A2, A6);
  w_gemm<n>(l, A6, A2, A8);
#pragma unroll
  for (int e0 = 0; e0 < nn; e0 += 64) {
    const int e = e0 + l < nn ? e0 + l : nn - 1;
    const double id = (e / n == e % n) ? 1.0 : 0.0, a2 = A2[e], a4 = A4[e], a6 = A6[e], a8 = A8[e];
    const double t = (((pade9(9) * a8 + pade9(7) * a6) + pade9(5) * a4) + pade9(3) * a2) + pade9(1) * id;
    const double v = (((pade9(8) * a8 + pade9(6) * a6) + pade9(4) * a4) + pade9(2) * a2) + pade9(0) * id;
    if (e0 + l < nn) {
      T[e] = t;
      V[e] = v;
      W[e] = a2;
    }
  }
  wave_sync();
  w_gemm<n>(l, Ap, T, A4);  // the odd part of the Pade approximant
  w_gemm_cols<n, d>(l, A2, Bp, PB);
  // the lane's column of the system
  const bool den = l < n, num_l = l >= n && l < 2 * n;
  const int mc = den ? l : (num_l ? l - n : n - 1);
  const int rc = l >= 2 * n ? (l - 2 * n < m10 ? l - 2 * n : m10 - 1) : 0, rk = rc % d;
  double x[n];
#pragma unroll
  for (int r = 0; r < n; ++r) x[r] = c.lg.c[1] * PB[r * d + rk] + c.lg.c[0] * Bp[r * d + rk];
  // the Legendre terms: blocks 2i (even) and 2i + 1 (odd)
#pragma unroll
  for (int kk = 2; kk <= 4; ++kk) {
    double* const to = kk % 2 == 0 ? T : W;
    w_gemm<n>(l, A2, kk % 2 == 0 ? W : T, to);
    w_gemm_cols<n, d>(l, to, Bp, PB);
#pragma unroll
    for (int r = 0; r < n; ++r) x[r] = x[r] + c.lg.c[kk] * PB[r * d + rk];
  }
  // L_odd = A L_odd, then every block / sqrt(2 b + 1)
  {
    const bool odd = (rc / d) % 2 == 1;
    double y[n];
#pragma unroll
    for (int r = 0; r < n; ++r) {
      double acc = 0.0;
#pragma unroll
      for (int q = 0; q < n; ++q) acc += Ap[r * n + q] * x[q];
      y[r] = acc;
    }
#pragma unroll
    for (int r = 0; r < n; ++r) {
      const double v = lane_div(odd ? y[r] : x[r], c.lg.den, c.lg.rden);
      const double vv = V[r * n + mc], pw = A4[r * n + mc], m = den ? vv - pw : vv + pw;
      x[r] = l < 2 * n ? m : v;
    }
  }
  wave_lu<n>(x, l);
  double sol[n];
  wave_backsolve<n>(x, l, sol);
  if (num_l)
#pragma unroll
    for (int i = 0; i < n; ++i) eA[i * n + mc] = sol[i];
  if (l >= 2 * n && l < 2 * n + m10)
#pragma unroll
    for (int i = 0; i < n; ++i) rhs[i * m10 + rc] = sol[i];
  wave_sync();
  const int row = w_row(c);
  {
    // qr_r(L^T)^T: the Gramian factor of the scaled problem
    double a[m10];
#pragma unroll
    for (int r = 0; r < m10; ++r) a[r] = rhs[row * m10 + r];
    wave_qr<WPatTall<SH>>(a, l);
    const int here = wave_here(row);
    if (l < n)
#pragma unroll
      for (int i = 0; i < n; ++i) U[row * n + i] = wave_r(a, i, here);
    wave_sync();
  }
  // _exp_gram_cholesky_double
  for (int it = 0; it < nd; ++it) {
    double a[2 * n];
#pragma unroll
    for (int r = 0; r < n; ++r) {
      a[r] = U[row * n + r];
      a[n + r] = 0.0;
    }
#pragma unroll
    for (int k = 0; k < n; ++k) {
      const double g = eA[row * n + k];
#pragma unroll
      for (int r = 0; r <= k; ++r) a[n + r] += g * U[k * n + r];
    }
    w_gemm<n>(l, eA, eA, T);
    wave_qr<WPatDouble<SH>>(a, l);
    const int here = wave_here(row);
    if (l < n)
#pragma unroll
      for (int i = 0; i < n; ++i) U[row * n + i] = wave_r(a, i, here);
    wave_copy<nn>(l, eA, T);
    wave_sync();
  }
  // non-negative diagonal (column signs)
  double sgn[n], u[n];
#pragma unroll
  for (int j = 0; j < n; ++j) {
    sgn[j] = U[j * n + j] < 0.0 ? -1.0 : 1.0;
    u[j] = U[row * n + j];
  }
  wave_sync();
  if (l < n)
#pragma unroll
    for (int j = 0; j < n; ++j) U[row * n + j] = u[j] * sgn[j];
  wave_sync();
}

template <class SH>
__device__ __forceinline__ double w_noise_scale(const WCtx<SH>& c, double dt, double s) {
  if (SH::expo) return s;  // the factor holds sqrt|dt| and the base scale
  if (SH::dense) return sqrt(fabs(dt)) * s;
  return sqrt(fabs(dt)) * c.a->cfg.base_output_scale * s;
}

// The entries A[i][k] of row i of the transition in ascending k: f(A[i][k], k).
template <class SH, class F>
__device__ __forceinline__ void w_prior_terms(const WCtx<SH>& c, int i, F f) {
  const int k0 = SH::st == 1 ? 0 : i % SH::st;
#pragma unroll
  for (int q = 0; q < SH::nc / SH::st; ++q) {
    const int k = q * SH::st + k0;
    f(c.A()[i * SH::nc + k], k);
  }
}

// Column i of (A (|p| * L))^T: a[r] = sum_k A[i][k] (|p_k| L[k][r]), L lower
// triangular (p is positive but for non-finite steps).
template <class SH>
__device__ __forceinline__ void w_prior_column(const WCtx<SH>& c, int i, const double* L, bool abs_p, double* a) {
  const int k0 = SH::st == 1 ? 0 : i % SH::st;
#pragma unroll
  for (int r = 0; r < SH::nc; ++r) a[r] = 0.0;
#pragma unroll
  for (int q = 0; q < SH::nc / SH::st; ++q) {
    const int k = q * SH::st + k0;
    const double ak = c.A()[i * SH::nc + k], p = c.PI()[k], pk = abs_p ? fabs(p) : p;
#pragma unroll
    for (int r = 0; r < (q + 1) * SH::st; ++r) a[r] += ak * (pk * L[k * SH::nc + r]);
  }
}

// apply_flat of the transition to a mean x: out = p * (A (p^-1 * x)) (dense)
// or (p * A) (p^-1 * x) (isotropic).
template <class SH>
__device__ __forceinline__ void w_apply_flat_mean(const WCtx<SH>& c, const double* x, double* out) {
  const int i = w_row(c);
  double acc[SH::mc] = {};
  w_prior_terms(c, i, [&](double ak, int k) {
#pragma unroll
    for (int col = 0; col < SH::mc; ++col) {
      if (SH::dense) acc[col] += ak * (c.PI()[k] * x[k * SH::mc + col]);
      else acc[col] += (c.P()[i] * ak) * (c.PI()[k] * x[k * SH::mc + col]);
    }
  });
  if (c.l < SH::nc)
#pragma unroll
    for (int col = 0; col < SH::mc; ++col)
      out[i * SH::mc + col] = SH::dense ? c.P()[i] * (acc[col] + 0.0) : acc[col] + 0.0;
  wave_sync();
}

// ts0 / ts1 linearisation at the mean Xm (ssm_impl_dense.py:237-334,
// ssm_impl_isotropic.py:298-355 with the exact trace).
template <class SH>
__device__ __forceinline__ void w_linearize(const WCtx<SH>& c, const double* Xm, double t, WLin<SH>& lin) {
  constexpr int d = SH::d, ko = SH::ko, K2 = 2 * SH::ko;
  const int id = c.cfg.vector_field;
  double y[d];
#pragma unroll
  for (int j = 0; j < d; ++j) y[j] = Xm[j];
  double f[d];
#pragma unroll
  for (int j = 0; j < d; ++j) f[j] = vf_component(id, d, y, c.prm(), t, j);
  if (!c.ts1()) {
#pragma unroll
    for (int j = 0; j < d; ++j) lin.b[j] = wave_rounded(-f[j]);
#pragma unroll
    for (int e = 0; e < ko * K2; ++e) lin.J[e] = 0.0;
    return;
  }
  if constexpr (SH::dense) {
#pragma unroll
    for (int i = 0; i < ko; ++i) {
#pragma unroll
      for (int j = 0; j < K2; ++j)
        lin.J[i * K2 + j] = j < d ? -vf_jac(id, d, y, c.prm(), i, j < d ? j : 0) : (j == d + i ? 1.0 : 0.0);
      double jm = 0.0;
#pragma unroll
      for (int k = 0; k < K2; ++k) jm += lin.J[i * K2 + k] * Xm[k];
      lin.b[i] = wave_rounded((Xm[d + i] - f[i]) - jm);
    }
  } else {
    double tr = 0.0;
#pragma unroll
    for (int j = 0; j < d; ++j) tr += -vf_jac(id, d, y, c.prm(), j, j);
    const double h0 = tr / (double)d;
    lin.J[0] = h0;
    lin.J[1] = 1.0;
#pragma unroll
    for (int j = 0; j < d; ++j) {
      const double r = Xm[d + j] - f[j];
      lin.b[j] = wave_rounded(r - (h0 * Xm[j] + Xm[d + j]));
    }
  }
}

// Entry (o, col) of H X for a mean X.
template <class SH>
__device__ __forceinline__ double w_hm(const WCtx<SH>& c, const WLin<SH>& lin, const double* X, int o, int col) {
  constexpr int K2 = 2 * SH::ko;
  if (!c.ts1()) return X[(SH::ko + o) * SH::mc + col];
  double acc = 0.0;
#pragma unroll
  for (int k = 0; k < K2; ++k) acc += lin.J[o * K2 + k] * X[k * SH::mc + col];
  return acc;
}

// Column r of row o (the lane's) of H L for a lower-triangular factor given by
// its entries L(k, r).
template <class SH, class LF>
__device__ __forceinline__ double w_hl(const WCtx<SH>& c, const WLin<SH>& lin, LF L, int o, int r) {
  constexpr int K2 = 2 * SH::ko;
  if (!c.ts1()) return L(SH::ko + o, r);
  double acc = 0.0;
#pragma unroll
  for (int k = 0; k < K2; ++k) {
    double j = lin.J[k];
#pragma unroll
    for (int q = 1; q < SH::ko; ++q) j = o == q ? lin.J[q * K2 + k] : j;
    acc += j * L(k, r);
  }
  return acc;
}

// residual_whitened_rms against zero data (ssm_impl_dense.py:156-160,
// isotropic :203-207) of an observed marginal held by every lane.
template <class SH>
__device__ __forceinline__ double w_rms_zero(const double* om, const double* oL) {
  constexpr int k = SH::ko, m = SH::mc;
  double sum[m];
#pragma unroll
  for (int col = 0; col < m; ++col) {
    double x[k], sq = 0.0;
#pragma unroll
    for (int i = 0; i < k; ++i) {
      double s = SH::dense ? (0.0 - om[i * m + col]) : om[i * m + col];
#pragma unroll
      for (int j = 0; j < i; ++j) s -= oL[i * k + j] * x[j];
      x[i] = s / oL[i * k + i];
      sq = wave_add_square(sq, x[i]);
    }
    sum[col] = sq;
  }
  double tot = sum[0];
  if constexpr (m == 2) tot = wave_add(sum[0], sum[1]);
  return wave_div_root<k * m>(sqrt(tot));
}

// The error model's observed marginal at the extrapolation Um with output
// scale 1 (fx.marginalise of (Um, |p| (s1 Q))): oL and sigma, in every lane.
template <class SH>
__device__ __forceinline__ void w_calibrate(const WCtx<SH>& c, const WLin<SH>& lin, const double* Um, double s1,
                                            WErr& err) {
  constexpr int k = SH::ko, m = SH::mc;
  const int o = c.l < k ? c.l : k - 1;
  const double damp = c.cfg.damp;
  double a[3 * k], om[k * m];
#pragma unroll
  for (int r = 0; r < 2 * k; ++r)
    a[r] = w_hl(c, lin, [&](int q, int col) { return wave_rounded(fabs(c.P()[q]) * (s1 * c.Q()[q * SH::nc + col])); }, o, r);
#pragma unroll
  for (int r = 0; r < k; ++r) a[2 * k + r] = r == o ? damp : 0.0;
#pragma unroll
  for (int i = 0; i < k; ++i)
#pragma unroll
    for (int col = 0; col < m; ++col) om[i * m + col] = w_hm(c, lin, Um, i, col) + lin.b[i * m + col];
  wave_qr<WPatFx<SH>>(a, c.l);
#pragma unroll
  for (int i = 0; i < k; ++i)
#pragma unroll
    for (int j = 0; j < k; ++j) err.oL[i * k + j] = j <= i ? wave_bcast(a[j], i) : 0.0;
  err.sigma = w_rms_zero<SH>(om, err.oL);
}

// marginalise of the transition (ssm_impl_dense.py:24-33, isotropic :81-89).
template <class SH>
__device__ __forceinline__ void w_marginalise_prior(const WCtx<SH>& c, double s, const double* Xm, const double* XL,
                                                    double* Ym, double* YL) {
  constexpr int n = SH::nc, m = SH::mc;
  const int i = w_row(c);
  double a[2 * n], acc[m] = {};
  w_prior_column(c, i, XL, false, a);
#pragma unroll
  for (int r = 0; r < n; ++r) a[n + r] = wave_rounded(s * c.Q()[i * n + r]);
  w_prior_terms(c, i, [&](double ak, int k) {
#pragma unroll
    for (int col = 0; col < m; ++col) acc[col] += ak * (c.PI()[k] * Xm[k * m + col]);
  });
  wave_qr<WPatStack<SH>>(a, c.l);
  const double p = c.P()[i];
  if (c.l < n) {
#pragma unroll
    for (int col = 0; col < m; ++col) Ym[i * m + col] = p * (acc[col] + 0.0);
    const int here = wave_here(i);
#pragma unroll
    for (int j = 0; j < n; ++j) YL[i * n + j] = fabs(p) * wave_r(a, j, here);
  }
  wave_sync();
}

// revert of the transition (ssm_impl_dense.py:51-77, isotropic :107-133,
// cholesky_util.py:27-82): X -> observed (Ym, YL) and backward conditional B.
template <class SH>
__device__ __forceinline__ void w_revert_prior(const WCtx<SH>& c, double s, const double* Xm, const double* XL,
                                               double* Ym, double* YL, double* B, double* tmp) {
  constexpr int n = SH::nc, m = SH::mc;
  // lanes 0..n-1: the left columns, lanes n..2n-1: the right ones (the others repeat the last)
  const bool right = c.l >= n;
  const int i = right ? (c.l < 2 * n ? c.l - n : n - 1) : c.l;
  double a[2 * n], acc[m] = {};
  const double p = c.P()[i], pi = c.PI()[i];
  {
    double left[n];
    w_prior_column(c, i, XL, true, left);
#pragma unroll
    for (int r = 0; r < n; ++r) {
      const double x = wave_rounded(fabs(pi) * XL[i * n + r]), q = wave_rounded(s * c.Q()[i * n + r]);
      a[r] = right ? 0.0 : q;
      a[n + r] = right ? x : left[r];
    }
  }
  // mean_observed = A (p^-1 * m)
  w_prior_terms(c, i, [&](double ak, int k) {
#pragma unroll
    for (int col = 0; col < m; ++col) acc[col] += ak * (c.PI()[k] * Xm[k * m + col]);
  });
  double xm[m];
#pragma unroll
  for (int col = 0; col < m; ++col) {
    xm[col] = Xm[i * m + col];
    if (!right) tmp[i * m + col] = acc[col] + 0.0;
  }
  wave_sync();
  wave_qr<WPatRevert<SH>>(a, c.l);
  // the gain's row i: back substitution of the right column with R_Y
  double gn[n];
  wave_backsolve<n>(a, c.l, gn);
  if (right && c.l < 2 * n) {
#pragma unroll
    for (int k = 0; k < n; ++k) B[SH::cA + i * n + k] = gn[k];
#pragma unroll
    for (int col = 0; col < m; ++col) {
      double ac = 0.0;
#pragma unroll
      for (int k = 0; k < n; ++k) ac += gn[k] * tmp[k * m + col];
      B[SH::cm + i * m + col] = pi * xm[col] - ac;
    }
    const int here = wave_here(i);
#pragma unroll
    for (int j = 0; j < n; ++j) B[SH::cL + i * n + j] = j <= here ? a[n + j] : 0.0;
    B[SH::ctl + i] = 1.0 / p;
    B[SH::cto + i] = 1.0 / pi;
  }
  if (!right) {
#pragma unroll
    for (int col = 0; col < m; ++col) Ym[i * m + col] = p * tmp[i * m + col];
    const int here = wave_here(i);
#pragma unroll
    for (int j = 0; j < n; ++j) YL[i * n + j] = fabs(p) * wave_r(a, j, here);
  }
  wave_sync();
}

// merge (ssm_impl_dense.py:35-49, isotropic :91-105): R = F o B, F possibly the
// identity (then exactly the rescaled B).  R may not share storage with F or B.
template <class SH>
__device__ __forceinline__ void w_merge(const WCtx<SH>& c, bool ident, const double* F, const double* B, double* R) {
  constexpr int n = SH::nc, m = SH::mc;
  const double *oA = B + SH::cA, *om = B + SH::cm, *oL = B + SH::cL, *oto = B + SH::cto;
  const int i = w_row(c);
  if (ident) {
#pragma unroll
    for (int e0 = 0; e0 < n * n; e0 += 64) {
      const int e = e0 + c.l;
      if (e < n * n) {
        const double T = 1.0 * oto[e / n];
        R[SH::cA + e] = T * oA[e];
        R[SH::cL + e] = fabs(T) * oL[e];
      }
    }
    if (c.l < n) {
#pragma unroll
      for (int col = 0; col < m; ++col) R[SH::cm + i * m + col] = (1.0 * oto[i]) * om[i * m + col] + 0.0;
      R[SH::ctl + i] = B[SH::ctl + i];
      R[SH::cto + i] = 1.0;
    }
    wave_sync();
    return;
  }
  const double *sA = F + SH::cA, *sm = F + SH::cm, *sL = F + SH::cL, *stl = F + SH::ctl;
  double a[2 * n], acc[m] = {};
#pragma unroll
  for (int r = 0; r < n; ++r) {
    a[r] = 0.0;
    a[n + r] = sL[i * n + r];  // R2 = C1^T
  }
  // R1 = (A1 (|T| o C2))^T with C2 lower triangular, and m = A1 (T o m2) + m1
#pragma unroll
  for (int k = 0; k < n; ++k) {
    const double T = stl[k] * oto[k], g = sA[i * n + k];
#pragma unroll
    for (int r = 0; r <= k; ++r) a[r] += g * (fabs(T) * oL[k * n + r]);
#pragma unroll
    for (int col = 0; col < m; ++col) acc[col] += g * (T * om[k * m + col]);
  }
  // A = A1 (T o A2), spread over all lanes
#pragma unroll
  for (int e0 = 0; e0 < n * n; e0 += 64) {
    const int e = e0 + c.l < n * n ? e0 + c.l : n * n - 1, ei = e / n, ej = e % n;
    double ac = 0.0;
#pragma unroll
    for (int k = 0; k < n; ++k) ac += sA[ei * n + k] * ((stl[k] * oto[k]) * oA[k * n + ej]);
    if (e0 + c.l < n * n) R[SH::cA + e] = ac;
  }
  wave_qr<WPatStack<SH>>(a, c.l);
  if (c.l < n) {
#pragma unroll
    for (int col = 0; col < m; ++col) R[SH::cm + i * m + col] = acc[col] + sm[i * m + col];
    const int here = wave_here(i);
#pragma unroll
    for (int j = 0; j < n; ++j) R[SH::cL + i * n + j] = wave_r(a, j, here);
    R[SH::ctl + i] = B[SH::ctl + i];
    R[SH::cto + i] = F[SH::cto + i];
  }
  wave_sync();
}

// marginalise of a backward conditional C (estimators_and_losses.py:156-178).
// Y may share storage with X: a lane reads its inputs before the QR.
template <class SH>
__device__ __forceinline__ void w_marginalise_cond(const WCtx<SH>& c, const double* C, const double* Xm,
                                                   const double* XL, double* Ym, double* YL) {
  constexpr int n = SH::nc, m = SH::mc;
  const int i = w_row(c);
  double a[2 * n], acc[m] = {};
#pragma unroll
  for (int r = 0; r < n; ++r) {
    a[r] = 0.0;
    a[n + r] = C[SH::cL + i * n + r];
  }
#pragma unroll
  for (int k = 0; k < n; ++k) {
    const double g = C[SH::cA + i * n + k], tl = C[SH::ctl + k];
#pragma unroll
    for (int r = 0; r <= k; ++r) a[r] += g * (tl * XL[k * n + r]);
#pragma unroll
    for (int col = 0; col < m; ++col) acc[col] += g * (tl * Xm[k * m + col]);
  }
  wave_sync();
  wave_qr<WPatStack<SH>>(a, c.l);
  const double to = C[SH::cto + i];
  if (c.l < n) {
#pragma unroll
    for (int col = 0; col < m; ++col) Ym[i * m + col] = to * (acc[col] + C[SH::cm + i * m + col]);
    const int here = wave_here(i);
#pragma unroll
    for (int j = 0; j < n; ++j) YL[i * n + j] = fabs(to) * wave_r(a, j, here);
  }
  wave_sync();
}

// fx.revert(pred) and apply_flat(data) (ssm_impl_api.py:112-132):
// (Pm, PL) -> (Xm, XL); `obs` receives the observed marginal's mean and factor.
template <class SH>
__device__ __forceinline__ void w_update(const WCtx<SH>& c, const WLin<SH>& lin, const double* Pm, const double* PL,
                                         double* Xm, double* XL, double* om, double* oL) {
  constexpr int n = SH::nc, k = SH::ko, m = SH::mc;
  const double damp = c.cfg.damp;
  // lanes 0..k-1: the observation's columns, lanes k..k+n-1: the state's (the others repeat the last)
  const bool state = c.l >= k;
  const int o = state ? k - 1 : c.l;
  const int i = state ? (c.l < k + n ? c.l - k : n - 1) : 0;
  double a[k + n];
#pragma unroll
  for (int r = 0; r < k; ++r) a[r] = !state && r == o ? damp : 0.0;
#pragma unroll
  for (int r = 0; r < n; ++r) {
    const double x = PL[i * n + r];
    double h = 0.0;
    if (r < 2 * k) h = w_hl(c, lin, [&](int q, int col) { return PL[q * n + col]; }, o, r);
    a[k + r] = state ? x : h;
  }
#pragma unroll
  for (int r = 0; r < k; ++r)
#pragma unroll
    for (int col = 0; col < m; ++col) om[r * m + col] = w_hm(c, lin, Pm, r, col) + lin.b[r * m + col];
  wave_qr<WPatUpdate<SH>>(a, c.l);
  double gn[k];
  wave_backsolve<k>(a, c.l, gn);
  if (state && c.l < k + n) {
#pragma unroll
    for (int col = 0; col < m; ++col) {
      double acc = 0.0;
#pragma unroll
      for (int r = 0; r < k; ++r) acc += gn[r] * om[r * m + col];
      Xm[i * m + col] = Pm[i * m + col] - acc;
    }
    const int here = wave_here(i);
#pragma unroll
    for (int j = 0; j < n; ++j) XL[i * n + j] = j <= here ? a[k + j] : 0.0;
  }
#pragma unroll
  for (int i2 = 0; i2 < k; ++i2)
#pragma unroll
    for (int j = 0; j < k; ++j) oL[i2 * k + j] = j <= i2 ? wave_bcast(a[j], i2) : 0.0;
  wave_sync();
}

// error_residual_std.estimate_error_norm (solvers.py:925-996); dtn = dt^nord.
// Lane k < d takes dimension k.
template <class SH>
__device__ __forceinline__ double w_error_power(const WCtx<SH>& c, const WErr& err, const double* prev_m,
                                                const double* prop_m, double dtn, int nord) {
  constexpr int k = SH::ko, d = SH::d;
  const WCfg& cfg = c.cfg;
  const int q = c.l < d ? c.l : d - 1;
  // std of the lane's rescaled observed row: dense per-row qr_r (|beta| of
  // dlarfg), isotropic vector_norm
  const int r = k == 1 ? 0 : q;
  double row[k];
#pragma unroll
  for (int j = 0; j < k; ++j) {
    row[j] = err.oL[j];
#pragma unroll
    for (int x = 1; x < k; ++x) row[j] = r == x ? err.oL[x * k + j] : row[j];
  }
  double ss = 0.0;
#pragma unroll
  for (int j = 1; j < k; ++j) {
    const double x = err.sigma * row[j];
    ss += x * x;
  }
  const double alpha = err.sigma * row[0];
  double std;
  if (SH::dense) std = ss == 0.0 ? fabs(alpha) : fabs(hypot(alpha, sqrt(ss)));
  else std = sqrt(alpha * alpha + ss);
  const double e = nord == 1 ? std * dtn : std * dtn * 0.5;  // / n!, exactly
  const double ref = fmax(fabs(prev_m[q]), fabs(prop_m[q]));
  double norm;
  if (cfg.error_norm == PDQ_NORM_SCALE_THEN_RMS) {
    const double rr = e / (cfg.atol + cfg.rtol * fabs(ref));
    double tot = 0.0;
#pragma unroll
    for (int x = 0; x < d; ++x) {
      const double rx = wave_bcast(rr, x);
      tot = wave_add_square(tot, rx);
    }
    norm = wave_div_root<d>(sqrt(tot));
  } else {
    double sa = 0.0, sr = 0.0;
#pragma unroll
    for (int x = 0; x < k; ++x) {
      const double ex = wave_bcast(e, x);
      sa = wave_add_square(sa, ex);
    }
#pragma unroll
    for (int x = 0; x < d; ++x) {
      const double rx = wave_bcast(ref, x);
      sr = wave_add_square(sr, rx);
    }
    norm = (sqrt(sa) / sqrt((double)k)) / (cfg.atol + cfg.rtol * (sqrt(sr) / sqrt((double)d)));
  }
  return pow(norm, -1.0 / (double)SH::N);
}

// controllers.py:66-84 / :24-63
template <class SH>
__device__ __forceinline__ double w_control(const WCtx<SH>& c, double dt, double& cstate, double ep) {
  const WCfg& cfg = c.cfg;
  if (cfg.integral) {
    const double ratio = cfg.safety * ep;
    return fmax(cfg.factor_min, fmin(ratio, cfg.factor_max)) * dt;
  }
  const double gi = pow(ep, c.a->cfg.exponent_integral);
  const double gp = pow(ep / cstate, c.a->cfg.exponent_proportional);
  const double ratio = cfg.safety * gi * gp;
  const double sf = fmax(cfg.factor_min, fmin(ratio, cfg.factor_max));
  if (ep >= 1.0) cstate = ep;
  return sf * dt;
}

// ---------------------------------------------------------------- outputs
template <class SH>
__device__ __forceinline__ void w_write_normal(const WCtx<SH>& c, const double* m, const double* L, double* gm,
                                               double* gL) {
  if (gm) wave_copy<SH::ms>(c.l, gm, m);
  if (gL) wave_copy<SH::nn>(c.l, gL, L);
}

// Checkpoint k: the filter's marginal, or the smoothers' filtering marginal
// and (C) the backward conditional that leads to it, an identity with `ident`.
template <class SH>
__device__ __forceinline__ void w_write_checkpoint(const WCtx<SH>& c, int k, double t, const double* m,
                                                   const double* L, double os, int nsteps, const double* C,
                                                   bool ident) {
  const auto& o = c.a->out;
  const int K = c.K;
  const size_t row = (size_t)c.inst * K + k;
  // the outputs' addresses in one batch of scalar loads
  double *gt = o.t, *gos = c.dynamic ? o.output_scale : nullptr;
  double *gm = SH::smoother ? o.filt_mean : o.mean, *gL = SH::smoother ? o.filt_chol : o.chol;
  int64_t* gn = o.num_steps;
#ifndef PDQ_HOST_EMU
  asm("" : "+s"(gt), "+s"(gos), "+s"(gm), "+s"(gL), "+s"(gn));
#endif
  if (c.l == 0) {
    if (gt) gt[row] = t;
    if (gos) gos[row] = os;
    if (gn && k > 0) gn[(size_t)c.inst * (K - 1) + k - 1] = nsteps;
  }
  if constexpr (!SH::smoother) {
    w_write_normal(c, m, L, gm ? gm + row * SH::ms : nullptr, gL ? gL + row * SH::nn : nullptr);
  } else {
    w_write_normal(c, m, L, gm ? gm + row * SH::ms : nullptr, gL ? gL + row * SH::nn : nullptr);
    if (k == 0 || !C) return;
    const size_t idx = (size_t)c.inst * (K - 1) + k - 1;
#pragma unroll
    for (int e0 = 0; e0 < SH::nn; e0 += 64) {
      const int e = e0 + c.l;
      if (e < SH::nn) {
        o.cond_A[idx * SH::nn + e] = ident ? (e / SH::nc == e % SH::nc ? 1.0 : 0.0) : C[SH::cA + e];
        o.cond_chol[idx * SH::nn + e] = ident ? 0.0 : C[SH::cL + e];
      }
    }
    if (c.l < SH::ms) o.cond_mean[idx * SH::ms + c.l] = ident ? 0.0 : C[SH::cm + c.l];
    if (c.l < SH::nc) {
      o.cond_tl[idx * SH::nc + c.l] = ident ? 1.0 : C[SH::ctl + c.l];
      o.cond_to[idx * SH::nc + c.l] = ident ? 1.0 : C[SH::cto + c.l];
    }
  }
}

// userfriendly_output + strategy.finalize (solvers.py:439-480, 601-633,
// 735-767; estimators_and_losses.py:380-391, 437-470).
template <class SH>
__device__ __forceinline__ void w_finalize(const WCtx<SH>& c, int sf, const WScal& S) {
  const auto& cfg = c.a->cfg;
  const auto& o = c.a->out;
  constexpr int cs = SH::nn, ms = SH::ms;
  const int K = c.a->K, Km1 = K - 1, inst = c.inst;
  __threadfence_block();
  wave_sync();
  double scale = 1.0;
  const bool mle = cfg.solver == PDQ_SOLVER_MLE;
  if (mle) {
    scale = S.mle_run;
    if (cfg.correct_asymptotic_underconfidence) {
      const double ns = (double)o.num_steps[(size_t)inst * Km1 + Km1 - 1];
      scale = scale / sqrt(ns);
    }
    if (o.output_scale && c.l == 0)
      for (int k = 0; k < Km1; ++k) o.output_scale[(size_t)inst * K + k] = scale;
  } else if (cfg.solver == PDQ_SOLVER && o.output_scale && c.l == 0) {
    for (int k = 0; k < Km1; ++k) o.output_scale[(size_t)inst * K + k] = 1.0;
  }
  if constexpr (!SH::smoother) {
    if (mle && o.chol)
      for (int e = c.l; e < K * cs; e += 64)
        o.chol[(size_t)inst * K * cs + e] = scale * o.chol[(size_t)inst * K * cs + e];
  } else {
    double* const X = c.slot(sf);
    if (mle) {
      for (int e = c.l; e < K * cs; e += 64)
        o.filt_chol[(size_t)inst * K * cs + e] = scale * o.filt_chol[(size_t)inst * K * cs + e];
      for (int e = c.l; e < Km1 * cs; e += 64)
        o.cond_chol[(size_t)inst * Km1 * cs + e] = scale * o.cond_chol[(size_t)inst * Km1 * cs + e];
      for (int e = c.l; e < cs; e += 64) {
        X[SH::sL + e] = scale * X[SH::sL + e];
        X[SH::sC + SH::cL + e] = scale * X[SH::sC + SH::cL + e];
      }
      __threadfence_block();
      wave_sync();
    }
    // rv_at_t1 = posterior1.conditional.marginalise(posterior1.marginal), then
    // the backward pass x_j = cond_j.marginalise(x_{j+1}), j = K-2 .. 0; the
    // marginal stays in the terminal slot (j = K - 1: the terminal one itself)
    double* const C = c.lds + SH::oB;
    for (int j = Km1; j >= 0; --j) {
      const bool term = j == Km1;
      if (!term) {
        const size_t idx = (size_t)inst * Km1 + j;
        wave_copy<cs>(c.l, C + SH::cA, o.cond_A + idx * cs);
        wave_copy<cs>(c.l, C + SH::cL, o.cond_chol + idx * cs);
        wave_copy<ms>(c.l, C + SH::cm, o.cond_mean + idx * ms);
        wave_copy<SH::nc>(c.l, C + SH::ctl, o.cond_tl + idx * SH::nc);
        wave_copy<SH::nc>(c.l, C + SH::cto, o.cond_to + idx * SH::nc);
        wave_sync();
      }
      if (!(term && S.ident))
        w_marginalise_cond(c, term ? X + SH::sC : C, X + SH::sm, X + SH::sL, X + SH::sm, X + SH::sL);
      const size_t row = (size_t)inst * K + j;
      if (term)
        w_write_normal(c, X + SH::sm, X + SH::sL, o.term_mean ? o.term_mean + (size_t)inst * ms : nullptr,
                       o.term_chol ? o.term_chol + (size_t)inst * cs : nullptr);
      w_write_normal(c, X + SH::sm, X + SH::sL, o.mean ? o.mean + row * ms : nullptr,
                     o.chol ? o.chol + row * cs : nullptr);
      wave_sync();
    }
  }
}

// ---------------------------------------------------------------- the solve
enum { WOP_STEP = 0, WOP_BEYOND1 = 1, WOP_BEYOND2 = 2, WOP_AT = 3 };

// One instance: the save_at loop of solvers_via_adaptive_steps.py:46-375 (or
// the fixed grid, :11-34 of solvers_via_fixed_steps.py) with
// solver_dynamic.step (solvers.py:549-599), solver.step (:702-733) or
// solver_mle.step (:395-437), and interpolate_fwd (:205-315).
template <class SH>
__device__ __forceinline__ void w_solve_instance(WCtx<SH> c) {
  constexpr int n = SH::nc;
  const int K = c.K, inst = c.inst, l = c.l;
  const double* ts = c.a->times + (size_t)inst * K;
  const bool grid = c.a->mode == MODE_FIXED_GRID;
  const bool dynamic = c.dynamic, mle = c.a->cfg.solver == PDQ_SOLVER_MLE;
  const bool fp = SH::smoother && c.a->cfg.strategy == PDQ_FIXEDPOINT;
  const int nord = c.a->cfg.error_per_unit_step ? 2 : 1;
  double* const Um = c.lds + SH::oUm;
  double* const Pm = c.lds + SH::oPm;
  double* const PL = c.lds + SH::oPL;
  double* const B = c.lds + SH::oB;
  double* const E = c.lds + SH::oE;
  for (int i = l; i < c.a->cfg.n_params; i += 64) c.lds[SH::oPrm + i] = c.a->params[(size_t)inst * c.a->cfg.n_params + i];
  // prior init: mean = tcoeffs, chol = init_std * I (from_mean_and_std)
  int sf = 0, ifr = 1, pr = 2;
  {
    double* const S = c.slot(sf);
    const double* tc = c.a->tcoeffs + (size_t)inst * SH::N * SH::d;
    wave_copy<SH::N * SH::d>(l, S + SH::sm, tc);
#pragma unroll
    for (int e0 = 0; e0 < SH::ssize - SH::sL; e0 += 64) {
      const int e = e0 + l;
      if (e < SH::ssize - SH::sL) {
        const bool diag = e < SH::nn && e / n == e % n;
        S[SH::sL + e] = diag ? (c.a->cfg.init_std_rows ? c.a->cfg.init_std_rows[e / n] : c.a->cfg.init_std) : 0.0;
      }
    }
    wave_sync();
    wave_copy<SH::ssize>(l, c.slot(ifr), S);
    wave_sync();
  }
  WScal F{}, S{}, R{};
  S.t = wave_rounded(ts[0]);
  S.os = wave_rounded(1.0);
  S.ident = SH::smoother;
  F = S;
  w_write_checkpoint(c, 0, S.t, c.slot(sf) + SH::sm, c.slot(sf) + SH::sL, 1.0, 0, nullptr, false);
  int attempts = 0, accepted = 0;
  int status = PDQ_STATUS_OK, att = 0, k = 1;
  bool second = false;
  double dt = wave_rounded(c.a->cfg.dt0_per_instance ? c.a->cfg.dt0_per_instance[inst] : c.a->cfg.dt0), cstate = 1.0;
  // the point being solved for, and the one after it (its load is a point ahead of its use)
  double t1 = wave_rounded(ts[1]), t_prev = S.t, t_ahead = ts[K > 2 ? 2 : 1];
  auto next_point = [&]() {
    ++k;
    t_prev = t1;
    t1 = wave_rounded(t_ahead);
    t_ahead = ts[k + 1 < K ? k + 1 : K - 1];
  };
  while (k < K && status == PDQ_STATUS_OK) {
    c.renew();
    const WCfg& cfg = c.cfg;
    int op;
    if (grid) op = WOP_STEP;
    else if (second) op = WOP_BEYOND2;
    else if (wave_true(S.t + cfg.eps < t1)) op = WOP_STEP;
    else op = wave_true(S.t > t1 + cfg.eps) ? WOP_BEYOND1 : WOP_AT;
    if (op == WOP_AT) {
      // interpolate_fwd_at_t1 (solvers.py:271-315)
      const double* const X = c.slot(sf);
      w_write_checkpoint(c, k, S.t, X + SH::sm, X + SH::sL, S.os, S.nsteps, X + SH::sC, S.ident);
      wave_copy<SH::ssize>(l, c.slot(ifr), X);
      wave_sync();
      if (fp) S.ident = true;
      F = S;
      next_point();
      continue;
    }
    double h;
    if (op == WOP_STEP) {
      h = grid ? t1 - t_prev : dt;
      if (!grid && cfg.clip_dt) h = fmin(h, t1 - S.t);
    } else {
      h = op == WOP_BEYOND1 ? t1 - F.t : S.t - t1;
    }
    const double tn = S.t + h;
    const double dtn = w_precon(c, h, nord);
    if constexpr (SH::expo) w_exp_transition(c, h);
    // the state that is predicted: step_from, interp_from, or the interpolated marginal
    const double* const Xs = op == WOP_STEP ? c.slot(sf) : c.slot(ifr);
    const double *const Xm = Xs + SH::sm, *const XL = Xs + SH::sL;
    WLin<SH> lin;
    WErr err;
    double scale = S.os;
    if (op == WOP_STEP) {
      scale = 1.0;
      if (dynamic) {
        w_apply_flat_mean(c, Xm, Um);
        w_linearize(c, Um, tn, lin);
        w_calibrate(c, lin, Um, w_noise_scale(c, h, 1.0), err);
        scale = wave_rounded(err.sigma);
      }
    }
    const double s = w_noise_scale(c, h, scale);
    if constexpr (!SH::smoother) {
      w_marginalise_prior(c, s, Xm, XL, Pm, PL);
    } else {
      // the prediction into (Pm, PL) and the conditional into B; in front of it
      // the fixed-point smoother merges the state's own conditional
      w_revert_prior(c, s, Xm, XL, Pm, PL, B, c.lds + SH::oTmp);
      double* const dst = op == WOP_STEP ? c.slot(pr) + SH::sC : (op == WOP_BEYOND1 ? E : c.slot(sf) + SH::sC);
      if (fp) {
        w_merge(c, op == WOP_BEYOND2 || (op == WOP_STEP ? S.ident : F.ident),
                (op == WOP_BEYOND1 ? c.slot(ifr) : c.slot(sf)) + SH::sC, B, dst);
      } else {
        wave_copy<SH::csize>(l, dst, B);
        wave_sync();
      }
    }
    if (op == WOP_STEP) {
      double* const Y = c.slot(pr);
      double om[SH::ko * SH::mc], oL[SH::ko * SH::ko];
      if (!dynamic) w_linearize(c, Pm, tn, lin);
      w_update(c, lin, Pm, PL, Y + SH::sm, Y + SH::sL, om, oL);
      R = S;
      R.t = tn;
      R.os = dynamic ? scale : (mle ? S.os : 1.0);
      R.nsteps = S.nsteps + 1;
      R.ident = false;
      R.mle_run = R.mle_n = 0.0;
      if (mle) {
        // bayes_rule_and_residual_whitened_rms_tree: observed = (mo, R_Y^T)
        const double nt = w_rms_zero<SH>(om, oL);
        const double nd = S.mle_n;
        const double x1 = sqrt(nd / (nd + 1)) * S.mle_run;
        const double x2 = sqrt(1 / (nd + 1)) * nt;
        R.mle_run = hypot(x1, x2);
        R.mle_n = nd + 1;
      }
      ++attempts;
      if (grid) {
        ++accepted;
        w_write_checkpoint(c, k, tn, Y + SH::sm, Y + SH::sL, R.os, R.nsteps, Y + SH::sC, false);
        wave_sync();
        const int tmp = sf;
        sf = pr;
        pr = tmp;
        S = R;
        next_point();
        continue;
      }
      if (!dynamic) {
        w_apply_flat_mean(c, Xm, Um);
        w_calibrate(c, lin, Um, w_noise_scale(c, h, 1.0), err);
      }
      const double ep = wave_rounded(w_error_power(c, err, Xm, Y + SH::sm, dtn, nord));
      dt = wave_rounded(w_control(c, h, cstate, ep));
      ++att;
      const bool accept = wave_true(ep >= 1.0);
      if (!wave_true(isfinite(ep) && isfinite(dt))) {
        status = PDQ_STATUS_NONFINITE;
      } else if (wave_true(accept ? R.t == S.t : dt == 0.0 || S.t + dt == S.t)) {
        status = PDQ_STATUS_DT_UNDERFLOW;  // rejected and dt cannot advance t, or accepted without advancing it
      } else if ((!accept && cfg.max_attempts > 0 && att >= cfg.max_attempts) || attempts >= kMaxTotalAttempts) {
        status = PDQ_STATUS_MAX_ATTEMPTS;
      } else if (accept) {
        ++accepted;
        att = 0;
        // interp_from <- step_from, step_from <- proposed
        const int old = ifr;
        ifr = sf;
        sf = pr;
        pr = old;
        F = S;
        S = R;
      }
    } else if (op == WOP_BEYOND1) {
      // interpolate_fwd (solvers.py:205-269): the marginal at t1 is the new
      // interp_from's, E the conditional that leads to it
      double* const X = c.slot(ifr);
      w_write_checkpoint(c, k, t1, Pm, PL, S.os, S.nsteps, SH::smoother ? E : nullptr, false);
      wave_copy<SH::ms>(l, X + SH::sm, Pm);
      wave_copy<SH::nn>(l, X + SH::sL, PL);
      if (SH::smoother && !fp) wave_copy<SH::csize>(l, X + SH::sC, E);
      wave_sync();
      F.t = t1;
      if (SH::smoother) {
        F.ident = fp;
        second = true;
      } else {
        next_point();
      }
    } else {
      S.ident = false;
      second = false;
      next_point();
    }
  }
  if (status == PDQ_STATUS_OK) w_finalize(c, sf, S);
  c.renew();
  const auto& o = c.a->out;
  if (l == 0) {
    if (o.attempts) o.attempts[inst] = attempts;
    if (o.accepted) o.accepted[inst] = accepted;
    if (o.status) o.status[inst] = status;
  }
}

// The transition into LDS; lanes of one wavefront.
template <class SH>
__device__ __forceinline__ void w_setup(WArgs& a, double* lds, int l) {
  if constexpr (SH::expo) {
    wave_copy<SH::d * SH::nc>(l, lds + SH::xD, a.cfg.prior_drift);
  } else {
    wave_copy<SH::nn>(l, lds + SH::oA, a.A);
    wave_copy<SH::nn>(l, lds + SH::oQ, a.Q);
  }
  wave_sync();
}

}  // namespace pdq
