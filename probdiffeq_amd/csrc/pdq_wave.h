// Householder QR of a small matrix held by one wavefront: lane j holds column
// j in registers, and every index, loop bound and zero is known at compile
// time.
//
// The cooperative kernel's own QR (g_qr_r, pdq_coop.hip) keeps the matrix in LDS
// with run-time bounds, and each of a reflector's 2 (m - i) dependent fused
// multiply-adds waits for its operands from LDS.  Here a reflector is read
// from the pivot lane's registers into scalar registers (v_readlane_b32) and
// applied by all lanes at once; rows that the matrix's structure makes zero
// are skipped.  The arithmetic is that of g_qr_r at 64 lanes per group, bit
// for bit for finite data: the squared norm of a reflector is added up in the
// order of the 64-lane butterfly's lane 0, the products in row order, and the
// skipped rows would add exact zeros.
#pragma once

#include "pdq_device.h"

namespace pdq {

// The value that lane `src` (the same in every lane) holds, in every lane.
__device__ __forceinline__ double wave_bcast(double v, int src) {
#ifdef PDQ_HOST_EMU
  return pdq_emu_shfl(v, src, 64);
#else
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)u, src);
  const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(u >> 32), src);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
#endif
}

// The whole number that lane `src` holds, as a scalar.
__device__ __forceinline__ int wave_pick(int v, int src) {
#ifdef PDQ_HOST_EMU
  return (int)pdq_emu_shfl((double)v, src, 64);
#else
  return __builtin_amdgcn_readlane(v, src);
#endif
}

// The value that lane I of each row of 16 lanes holds, in that row's lanes: one
// instruction where wave_bcast takes two.
template <int I>
__device__ __forceinline__ double wave_bcast_row(double v) {
  static_assert(I < 16, "a lane of a row");
#ifdef PDQ_HOST_EMU
  return pdq_emu_shfl(v, I, 16);
#else
  return __builtin_amdgcn_update_dpp(0.0, v, 0x150 + I, 0xf, 0xf, true);  // row_newbcast
#endif
}

// The lane index as a value of its own: comparisons with it are made where
// they stand (one instruction) instead of ahead of the solve's loop, where
// their masks would take scalar registers throughout and be spilled.
__device__ __forceinline__ int wave_here(int lane) {
#ifndef PDQ_HOST_EMU
  asm("" : "+v"(lane));
#endif
  return lane;
}

// Whether v != 0 (or NaN) in lane src: a wave-uniform condition.
__device__ __forceinline__ bool wave_nonzero(double v, int src) {
#ifdef PDQ_HOST_EMU
  return wave_bcast(v, src) != 0.0;
#else
  return (__builtin_amdgcn_ballot_w64(v != 0.0) >> src) & 1;
#endif
}

// A matrix pattern Pat gives
//   COLS             columns (lanes that hold one)
//   M                rows held (a lane's registers)
//   NP               columns to triangularise (pivots 0..NP-1)
//   MROWS            rows of the whole matrix
//   row(r)           the matrix row that register r holds (ascending)
//   nz(r, c)         whether entry (register row r, column c) can be non-zero
// WaveQrPlan derives, per pivot i, the register rows its reflector touches
// (the rows below the pivot with a possibly non-zero entry in the pivot's
// column, fill-in of the earlier reflectors included), and the butterfly's
// positions that hold a value: bit p of has[i][L] for lane p after the
// strides 32 .. 2^L (a row at distance p + 1 below the pivot is lane p's).
template <class Pat>
struct WaveQrPlan {
  bool act[Pat::NP][Pat::M];
  bool any[Pat::NP];
  int piv[Pat::NP];  // the register row of the pivot
  uint64_t has[Pat::NP][7];

  constexpr WaveQrPlan() : act{}, any{}, piv{}, has{} {
    bool nz[Pat::M][Pat::NP] = {};
    for (int r = 0; r < Pat::M; ++r)
      for (int c = 0; c < Pat::NP; ++c) nz[r][c] = Pat::nz(r, c);
    for (int i = 0; i < Pat::NP; ++i) {
      piv[i] = 0;
      for (int r = 0; r < Pat::M; ++r)
        if (Pat::row(r) == i) piv[i] = r;
      if (Pat::MROWS - i <= 1) continue;
      for (int r = 0; r < Pat::M; ++r)
        if (Pat::row(r) > i && nz[r][i]) {
          act[i][r] = any[i] = true;
          has[i][6] |= uint64_t(1) << (Pat::row(r) - i - 1);
        }
      if (!any[i]) continue;
      for (int L = 5; L >= 0; --L)
        has[i][L] = (has[i][L + 1] | (has[i][L + 1] >> (1 << L))) & ((uint64_t(1) << (1 << L)) - 1);
      for (int c = i + 1; c < Pat::NP; ++c) {
        bool u = nz[piv[i]][c];
        for (int r = 0; r < Pat::M; ++r) u = u || (act[i][r] && nz[r][c]);
        nz[piv[i]][c] = u;
        for (int r = 0; r < Pat::M; ++r)
          if (act[i][r]) nz[r][c] = u;
      }
    }
  }
};

template <class Pat>
struct WaveQr {
  static_assert(Pat::MROWS <= 64, "one butterfly position per row");
  static constexpr WaveQrPlan<Pat> plan{};
  static constexpr int W = Pat::MROWS <= 16 ? 16 : (Pat::MROWS <= 32 ? 32 : 64);  // butterfly positions
  static constexpr int LW = W == 16 ? 4 : (W == 32 ? 5 : 6);

  // Lane 0's total of the butterfly over reflector I's squares.
  template <int I>
  static __device__ __forceinline__ double norm2(const double (&a)[Pat::M]) {
#ifdef __clang__
#pragma clang fp contract(off)  // the squares are rounded before the sums, as the butterfly's are
#endif
    double t[W];
#pragma unroll
    for (int r = 0; r < Pat::M; ++r)
      if (plan.act[I][r]) t[Pat::row(r) - I - 1] = a[r] * a[r];
#pragma unroll
    for (int L = LW - 1; L >= 0; --L)
#pragma unroll
      for (int p = 0; p < (1 << L); ++p) {
        const bool lo = (plan.has[I][L + 1] >> p) & 1, hi = (plan.has[I][L + 1] >> (p + (1 << L))) & 1;
        if (lo && hi) t[p] = t[p] + t[p + (1 << L)];
        else if (hi) t[p] = t[p + (1 << L)];
      }
    return t[0];
  }

  // A reflector's value in every lane that holds a column.
  template <int I>
  static __device__ __forceinline__ double bcast(double v) {
    if constexpr (Pat::COLS <= 16) return wave_bcast_row<I>(v);
    else return wave_bcast(v, I);
  }

  // Reflector I and the ones after it.
  template <int I>
  static __device__ __forceinline__ void from(double (&a)[Pat::M], int lane) {
    if constexpr (I < Pat::NP) {
      if constexpr (plan.any[I]) {
        constexpr int p = plan.piv[I];
        const double ss = norm2<I>(a);
        if (wave_nonzero(ss, I)) {
          const double alpha = a[p];
          const double beta = -copysign(lane_sqrt_pos(fma(alpha, alpha, ss)), alpha);
          const double tau = bcast<I>(lane_div_nz(beta - alpha, beta, lane_rcp_nz(beta)));
          const double scal = lane_rcp_nz(alpha - beta);
          double v[Pat::M];
#pragma unroll
          for (int r = 0; r < Pat::M; ++r)
            if (plan.act[I][r]) v[r] = bcast<I>(a[r] * scal);
          double w = alpha;
#pragma unroll
          for (int r = 0; r < Pat::M; ++r)
            if (plan.act[I][r]) w += v[r] * a[r];
          w *= tau;
          a[p] = wave_here(lane) == I ? beta : alpha - w;
#pragma unroll
          for (int r = 0; r < Pat::M; ++r)
            if (plan.act[I][r]) a[r] -= v[r] * w;
        }
      }
      from<I + 1>(a, lane);
    }
  }
};

// The QR in place: on return lane j's registers hold R's column j in the rows
// up to j; what the rows below hold is not meaningful (they are zero in R:
// read them through wave_r).
template <class Pat>
__device__ __forceinline__ void wave_qr(double (&a)[Pat::M], int lane) {
  WaveQr<Pat>::template from<0>(a, lane);
}

// Row r of R's column `col` from the registers wave_qr left.
template <int M>
__device__ __forceinline__ double wave_r(const double (&a)[M], int r, int col) {
  return r <= col ? a[r] : 0.0;
}

// x as a rounded value of its own: a product is not fused into the sums that
// take it (the run-time-shape kernel stores such products in LDS).
__device__ __forceinline__ double wave_rounded(double x) {
#ifndef PDQ_HOST_EMU
  asm("" : "+v"(x));
#endif
  return x;
}

// Whether c holds (the same in every lane), as a scalar condition: the branches
// on it are scalar ones, while the values it compares stay in vector registers
// (scalar registers are the scarce ones here).
__device__ __forceinline__ bool wave_true(bool c) {
#ifdef PDQ_HOST_EMU
  return c;
#else
  return __builtin_amdgcn_ballot_w64(c) != 0;
#endif
}

// acc + x x as one fused operation, also from acc = 0 (an addition of zero that
// is folded away would leave two products to choose from).
__device__ __forceinline__ double wave_add_square(double acc, double x) {
#ifdef PDQ_HOST_EMU
  return acc + x * x;
#else
  return wave_rounded(fma(x, x, acc));
#endif
}

// x + y, rounded on its own (neither a product of x nor of y is fused in).
__device__ __forceinline__ double wave_add(double x, double y) {
#ifdef __clang__
#pragma clang fp contract(off)
#endif
  return x + y;
}

// x / sqrt(n) for n = 1, 2: the division's quotient, from the constant's
// correctly rounded reciprocal (lane_div).
template <int n>
__device__ __forceinline__ double wave_div_root(double x) {
  static_assert(n == 1 || n == 2, "the roots of 1 and 2");
  constexpr double root = 1.4142135623730951, inverse = 0.7071067811865475;  // 1 / root, rounded to nearest
  return n == 1 ? x : lane_div(x, root, inverse);
}

// A whole number that every lane holds alike, as a scalar.
__device__ __forceinline__ int wave_int(int v) {
#ifdef PDQ_HOST_EMU
  return v;
#else
  return __builtin_amdgcn_readfirstlane(v);
#endif
}

// LU with partial pivoting (the first largest |entry| of each column pivots, as
// LAPACK's idamax) of the K x K matrix whose columns lanes 0..K-1 hold, with
// the row swaps and the forward substitution applied to the columns of all the
// other lanes: on return lane c < K holds U's column c in the rows up to c, the
// others their right-hand side, ready for wave_backsolve.
template <int K>
__device__ __forceinline__ void wave_lu(double (&a)[K], int lane) {
#pragma unroll
  for (int k = 0; k < K; ++k) {
    double best = -1.0;
    int bi = k;
#pragma unroll
    for (int r = k; r < K; ++r) {
      const double v = fabs(a[r]);
      if (v > best) {
        best = v;
        bi = r;
      }
    }
    const int piv = wave_pick(bi, k);
    if (piv != k) {
#pragma unroll
      for (int r = k + 1; r < K; ++r)
        if (piv == r) {
          const double t = a[k];
          a[k] = a[r];
          a[r] = t;
        }
    }
    const double inv = 1.0 / a[k];
#pragma unroll
    for (int r = k + 1; r < K; ++r) a[r] -= wave_bcast(a[r] * inv, k) * a[k];
  }
}

// Back substitution with the K x K leading triangle of R (lane c holds its
// column c): x = R^-1 a[0..K-1] for the lane's own column.  The quotients are
// those of the division: the diagonal's reciprocals are taken by their lanes
// at once and corrected against each residual (lane_div).
template <int K, int M>
__device__ __forceinline__ void wave_backsolve(const double (&a)[M], int lane, double (&x)[K]) {
  double dg = a[0];
  lane = wave_here(lane);
#pragma unroll
  for (int i = 1; i < K; ++i) dg = lane == i ? a[i] : dg;
  const double y = 1.0 / dg;
#pragma unroll
  for (int i = K - 1; i >= 0; --i) {
    double s = a[i];
#pragma unroll
    for (int c = i + 1; c < K; ++c) s -= wave_bcast(a[i], c) * x[c];
    x[i] = lane_div(s, wave_bcast(dg, i), wave_bcast(y, i));
  }
}

}  // namespace pdq
