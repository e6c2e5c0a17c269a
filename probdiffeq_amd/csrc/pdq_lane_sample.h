// Samples of a smoother's posterior (MarkovSequence.sample,
// estimators_and_losses.py:233-273), isotropic, one lane per (instance,
// sample).
//
// The reverse scan starts from a draw of the terminal marginal and pushes
// each sample back through the backward conditionals: predicted =
// cond.apply_flat(x), x = predicted.sample_flat(z).  The isotropic forms are
// kept exactly (ssm_impl_isotropic.py:75-79, 255-258): apply_flat adds the
// noise mean without the to_observed scaling the dense form applies, and
// sample_flat draws one N-vector z that every one of the d columns shares.
// The standard normal draws come in as data (the reference draws them from
// JAX keys): base[instance, sample, k] for conditional k, row K - 1 for the
// terminal marginal.
#pragma once

#include "pdq_lane.h"

namespace pdq {

// n doubles (8-byte aligned) from or to global memory, two per instruction.
struct alignas(8) SamplePair {
  double v[2];
};
// the same as a vector, for stores that leave the L2 to the reads
typedef double SampleVec __attribute__((vector_size(16), aligned(8)));
template <int n>
__device__ __forceinline__ void sample_load(const double* __restrict__ src, double* dst) {
#pragma unroll
  for (int e = 0; e + 1 < n; e += 2) {
    const SamplePair p = *reinterpret_cast<const SamplePair*>(src + e);
    dst[e] = p.v[0];
    dst[e + 1] = p.v[1];
  }
  if (n % 2) dst[n - 1] = src[n - 1];
}
template <int n>
__device__ __forceinline__ void sample_store(double* __restrict__ dst, const double* src) {
#pragma unroll
  for (int e = 0; e + 1 < n; e += 2) *reinterpret_cast<SamplePair*>(dst + e) = SamplePair{{src[e], src[e + 1]}};
  if (n % 2) dst[n - 1] = src[n - 1];
}

// One step of the scan: conditional k.
template <int N, int D>
struct SampleStep {
  double A[N * N], nm[N * D], nL[N * N], tl[N], to[N];
  __device__ __forceinline__ void load(const SampleArgs& a, size_t ci) {
    sample_load<N * N>(a.cond_A + ci * N * N, A);
    sample_load<N * D>(a.cond_mean + ci * N * D, nm);
    sample_load<N * N>(a.cond_chol + ci * N * N, nL);
    sample_load<N>(a.cond_tl + ci * N, tl);
    sample_load<N>(a.cond_to + ci * N, to);
  }
  // x <- the sample at k from the sample x at k + 1 and the draws z
  __device__ __forceinline__ void apply(const double* z, double* x) const {
    double xl[N * D], y[N * D];
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
      for (int c = 0; c < D; ++c) xl[i * D + c] = tl[i] * x[i * D + c];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const double toi = to[i];
      double lz = 0.0;
#pragma unroll
      for (int j = 0; j < N; ++j) lz += (fabs(toi) * nL[i * N + j]) * z[j];
#pragma unroll
      for (int c = 0; c < D; ++c) {
        double acc = 0.0;
#pragma unroll
        for (int j = 0; j < N; ++j) acc += (toi * A[i * N + j]) * xl[j * D + c];
        y[i * D + c] = (acc + nm[i * D + c]) + lz;
      }
    }
#pragma unroll
    for (int e = 0; e < N * D; ++e) x[e] = y[e];
  }
};

// The samples from the terminal marginal's draw: x at K - 1.
template <int N, int D>
__device__ __forceinline__ void lane_sample_terminal(const SampleArgs& a, size_t inst, const double* zk, double* x) {
  const double* m = a.term_mean + inst * N * D;
  const double* L = a.term_chol + inst * N * N;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    double acc = 0.0;
#pragma unroll
    for (int j = 0; j < N; ++j) acc += L[i * N + j] * zk[j];
#pragma unroll
    for (int c = 0; c < D; ++c) x[i * D + c] = m[i * D + c] + acc;
  }
}

// Steps k, k - 1, ... end of a lane's scan with the lane's own loads and
// (with `store`) stores.
template <int N, int D>
__device__ __forceinline__ void lane_sample_steps(const SampleArgs& a, size_t c0, int k, int end,
                                                  const double* __restrict__ z, double* __restrict__ out, double* x,
                                                  bool store = true) {
  for (; k >= end; --k) {
    SampleStep<N, D> s;
    s.load(a, c0 + k);
    s.apply(z + (size_t)k * N, x);
    if (store) sample_store<N * D>(out + (size_t)k * N * D, x);
  }
}

// One wavefront's 64 samples, kSampleTile points at a time.  What bounds the
// scan is memory: it reads the draws and writes the samples once, but a lane's
// own accesses to them are rows apart (a cache line per lane and instruction,
// fetched again for every point that shares it), and the scan is one
// dependent step per point with one wavefront per SIMD.  So the wavefront
// reads a tile of draws and writes a tile of samples row by row together,
// through LDS (rows of an odd number of doubles: a lane's column falls on
// banks of its own; a point's draws lie where its sample will).  With STAGED
// it also reads the conditionals of a tile together, one instance after the
// other, instead of every lane all 70 doubles of its instance's: at most
// kSampleInstances instances then share a wavefront, hence kSampleStagedMin
// samples.  Otherwise every lane loads its conditional, a step ahead into a
// second set of registers; all other loads are issued a tile ahead.
// 4096 instances x 16 samples x 200 points, nu = 4 (2.0 GB): 1.50 ms with a
// lane's loads at their use, 1.03 with them a step ahead, 0.68 with the tiles,
// 0.55 with tiles that begin at multiples of kSampleTile points (whole 64-byte
// sectors), 0.49 (4.2 TB/s; a large copy reaches 4.8) with stores that leave
// the L2 to the reads.  With 4 samples 0.81 -> 0.30 ms.
constexpr int kSampleTile = 4;
constexpr int kSampleInstances = 5;
constexpr int kSampleStagedMin = 16;  // 64 consecutive rows of >= 16 per instance meet at most 5 instances
static_assert((64 - 2) / kSampleStagedMin + 2 <= kSampleInstances, "instances of a wavefront");

// n pairs per row over 64 rows, as accesses f(q, row of access q in lane 0,
// the lane's row offset, the lane's pair): lanes side by side along a row, so
// that an access's address is a uniform part and one lane part.
template <int n, class F>
__device__ __forceinline__ void sample_pairs(int l, F&& f) {
  constexpr int a = n >= 16 ? 16 : 8, b = n - a;  // (n = 8, 10, 16, 20)
  static_assert(a <= n && (b == 0 || (b & (b - 1)) == 0), "two powers of two");
#pragma unroll
  for (int q = 0; q < a; ++q) f(q, q * (64 / a), l / a, l % a);
  if constexpr (b > 0) {
#pragma unroll
    for (int q = 0; q < b; ++q) f(a + q, q * (64 / b), l / b, a + l % b);
  }
}

template <int N, int D, bool STAGED>
struct SampleTile {
  static constexpr int zp = kSampleTile * N / 2, op = kSampleTile * N * D / 2;  // pairs per row
  static constexpr int os = kSampleTile * N * D + 1;                            // doubles of a row in LDS
  // the conditionals of a tile, one instance
  static constexpr int cA = 0, cL = cA + kSampleTile * N * N, cm = cL + kSampleTile * N * N,
                       ctl = cm + kSampleTile * N * D, cto = ctl + kSampleTile * N, csize = cto + kSampleTile * N;
  static constexpr int pA = kSampleTile * N * N / 2, pm = kSampleTile * N * D / 2, pt = kSampleTile * N / 2;
  static constexpr int lds = 64 * os + (STAGED ? kSampleInstances * csize : 0);  // doubles
  static_assert(kSampleTile % 2 == 0, "pairs, and two sets of registers");
  static_assert(pA <= 64 && pm + 2 * pt <= 64, "a lane per pair");
};

template <int N, int D, bool STAGED>
__device__ __forceinline__ void wave_sample(const SampleArgs& a, size_t g0, int rows, double* lds) {
  using T = SampleTile<N, D, STAGED>;
  constexpr int ND = N * D, NN = N * N;
  const int K = a.K, l = threadIdx.x;
  const size_t gid = g0 + (l < rows ? l : rows - 1);  // lanes without a sample repeat the last one
  const size_t inst = gid / (size_t)a.n_samples, c0 = inst * (size_t)(K - 1);
  const double* __restrict__ z = a.base + gid * K * N;
  double* __restrict__ out = a.samples + gid * K * ND;
  double* const row = lds + l * T::os;
  // draws of points k0 .. k0 + kSampleTile - 1 (rows beyond `rows` are not read)
  SamplePair zr[T::zp];
#pragma unroll
  for (int q = 0; q < T::zp; ++q) zr[q] = SamplePair{{0.0, 0.0}};
  auto load_draws = [&](int k0) {
    sample_pairs<T::zp>(l, [&](int q, int r0, int r, int p) {
      const double* const src = a.base + ((g0 + r0) * K + k0) * N;
      if (r0 + r < rows) zr[q] = *reinterpret_cast<const SamplePair*>(src + ((size_t)r * K * N + 2 * p));
    });
  };
  // STAGED: the conditionals of those points, instance first + i in cr[i]
  const size_t first = g0 / (size_t)a.n_samples;
  const int ni = (int)((g0 + rows - 1) / (size_t)a.n_samples - first) + 1;
  SamplePair cr[STAGED ? kSampleInstances : 1][3];
  auto load_conds = [&](int k0) {
#pragma unroll
    for (int i = 0; i < kSampleInstances; ++i)
      if (i < ni) {
        const size_t ci = (first + i) * (size_t)(K - 1) + k0;
        if (l < T::pA) {
          cr[i][0] = *reinterpret_cast<const SamplePair*>(a.cond_A + ci * NN + 2 * l);
          cr[i][1] = *reinterpret_cast<const SamplePair*>(a.cond_chol + ci * NN + 2 * l);
        }
        const double* const src = l < T::pm           ? a.cond_mean + ci * ND + 2 * l
                                  : l < T::pm + T::pt ? a.cond_tl + ci * N + 2 * (l - T::pm)
                                                      : a.cond_to + ci * N + 2 * (l - T::pm - T::pt);
        if (l < T::pm + 2 * T::pt) cr[i][2] = *reinterpret_cast<const SamplePair*>(src);
      }
  };
  SampleStep<N, D> s0, s1;
  // whole tiles down to point 0 (their rows then start at multiples of
  // kSampleTile points: whole 64-byte sectors where a row's length is one); the
  // points above them one by one
  int k = (K - 1) / kSampleTile * kSampleTile - 1;
  if (k > 0) {
    load_draws(k + 1 - kSampleTile);
    if constexpr (STAGED) load_conds(k + 1 - kSampleTile);
  }
  double x[ND];
  lane_sample_terminal<N, D>(a, inst, z + (size_t)(K - 1) * N, x);
  if (l < rows) sample_store<ND>(out + (size_t)(K - 1) * ND, x);
  lane_sample_steps<N, D>(a, c0, K - 2, k + 1, z, out, x, l < rows);
  if constexpr (!STAGED) {
    if (k > 0) s0.load(a, c0 + k);
  }
  for (; k > 0; k -= kSampleTile) {
    const int k0 = k + 1 - kSampleTile;
    const bool more = k0 > 0;
    sample_pairs<T::zp>(l, [&](int q, int r0, int r, int p) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int e = 2 * p + h;
        lds[r0 * T::os + (r * T::os + (e / N) * ND + e % N)] = zr[q].v[h];
      }
    });
    if constexpr (STAGED) {
#pragma unroll
      for (int i = 0; i < kSampleInstances; ++i)
        if (i < ni) {
          double* const dst = lds + 64 * T::os + i * T::csize;
          if (l < T::pA) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              dst[T::cA + 2 * l + h] = cr[i][0].v[h];
              dst[T::cL + 2 * l + h] = cr[i][1].v[h];
            }
          }
          if (l < T::pm + 2 * T::pt) {
#pragma unroll
            for (int h = 0; h < 2; ++h) dst[T::cm + 2 * l + h] = cr[i][2].v[h];
          }
        }
    }
    Grp<64>{}.sync();
    if (more) {
      load_draws(k0 - kSampleTile);
      if constexpr (STAGED) load_conds(k0 - kSampleTile);
    }
#pragma unroll
    for (int s = 0; s < kSampleTile; ++s) {
      const int t = kSampleTile - 1 - s;  // the point within the tile
      double zk[N];
#pragma unroll
      for (int j = 0; j < N; ++j) zk[j] = row[t * ND + j];
      if constexpr (STAGED) {
        const double* const c = lds + 64 * T::os + (int)(inst - first) * T::csize;
#pragma unroll
        for (int e = 0; e < NN; ++e) {
          s0.A[e] = c[T::cA + t * NN + e];
          s0.nL[e] = c[T::cL + t * NN + e];
        }
#pragma unroll
        for (int e = 0; e < ND; ++e) s0.nm[e] = c[T::cm + t * ND + e];
#pragma unroll
        for (int e = 0; e < N; ++e) {
          s0.tl[e] = c[T::ctl + t * N + e];
          s0.to[e] = c[T::cto + t * N + e];
        }
        s0.apply(zk, x);
      } else {
        const int next = k - s >= 1 ? k - s - 1 : 0;  // (the scan's last step loads conditional 0 again)
        if (s % 2) s0.load(a, c0 + next);
        else s1.load(a, c0 + next);
        if (s % 2) s1.apply(zk, x);
        else s0.apply(zk, x);
      }
#pragma unroll
      for (int j = 0; j < ND; ++j) row[t * ND + j] = x[j];
    }
    Grp<64>{}.sync();
    sample_pairs<T::op>(l, [&](int, int r0, int r, int p) {
      double* const dst = a.samples + ((g0 + r0) * K + k0) * ND;
      const double* const src = lds + r0 * T::os + (r * T::os + 2 * p);
      if (r0 + r < rows)
        __builtin_nontemporal_store(SampleVec{src[0], src[1]}, reinterpret_cast<SampleVec*>(dst + ((size_t)r * K * ND + 2 * p)));
    });
    Grp<64>{}.sync();
  }
}

template <int N, int D, bool STAGED>
__global__ void __launch_bounds__(64) lane_sample_kernel(SampleArgs a) {
  __shared__ double lds[SampleTile<N, D, STAGED>::lds];
  const size_t total = (size_t)a.n_inst * a.n_samples;
  const size_t stride = (size_t)gridDim.x * 64;
  for (size_t g = (size_t)blockIdx.x * 64; g < total; g += stride)
    wave_sample<N, D, STAGED>(a, g, (int)(total - g < 64 ? total - g : 64), lds);
}

}  // namespace pdq
