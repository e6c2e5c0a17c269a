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

// What one step of the scan reads: conditional k and the sample's draws.
template <int N, int D>
struct SampleStep {
  double A[N * N], nm[N * D], nL[N * N], tl[N], to[N], z[N];
  __device__ __forceinline__ void load(const SampleArgs& a, size_t ci, const double* __restrict__ zk) {
    sample_load<N * N>(a.cond_A + ci * N * N, A);
    sample_load<N * D>(a.cond_mean + ci * N * D, nm);
    sample_load<N * N>(a.cond_chol + ci * N * N, nL);
    sample_load<N>(a.cond_tl + ci * N, tl);
    sample_load<N>(a.cond_to + ci * N, to);
    sample_load<N>(zk, z);
  }
  // x <- the sample at k from the sample x at k + 1
  __device__ __forceinline__ void apply(double* x) const {
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

// The scan is one dependent step per point, and a batch of a few thousand
// instances gives each SIMD a single wavefront, so nothing but the lane's own
// loads can cover their latency: step k - 1's conditional and draws are
// loaded into a second set of registers before step k is computed, and two
// doubles move per instruction (a wavefront's lanes are 64 rows apart in the
// draws and samples: each access costs a cache line per lane).
// 4096 instances x 16 samples x 200 points, nu = 4: 1.49 -> 1.03 ms (2.0 GB).
template <int N, int D>
__device__ __forceinline__ void lane_sample(const SampleArgs& a, size_t gid) {
  const int K = a.K;
  const size_t inst = gid / (size_t)a.n_samples, c0 = inst * (size_t)(K - 1);
  const double* __restrict__ z = a.base + gid * K * N;
  double* __restrict__ out = a.samples + gid * K * N * D;
  double x[N * D];
  SampleStep<N, D> s0, s1;
  s0.load(a, c0 + K - 2, z + (size_t)(K - 2) * N);
  {
    const double* m = a.term_mean + inst * N * D;
    const double* L = a.term_chol + inst * N * N;
    const double* zk = z + (size_t)(K - 1) * N;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      double acc = 0.0;
#pragma unroll
      for (int j = 0; j < N; ++j) acc += L[i * N + j] * zk[j];
#pragma unroll
      for (int c = 0; c < D; ++c) x[i * D + c] = m[i * D + c] + acc;
    }
    sample_store<N * D>(out + (size_t)(K - 1) * N * D, x);
  }
  int k = K - 2;
  for (; k >= 1; k -= 2) {
    s1.load(a, c0 + k - 1, z + (size_t)(k - 1) * N);
    s0.apply(x);
    sample_store<N * D>(out + (size_t)k * N * D, x);
    const int next = k >= 2 ? k - 2 : 0;  // (the last pass loads conditional 0 again)
    s0.load(a, c0 + next, z + (size_t)next * N);
    s1.apply(x);
    sample_store<N * D>(out + (size_t)(k - 1) * N * D, x);
  }
  if (k == 0) {
    s0.apply(x);
    sample_store<N * D>(out, x);
  }
}

#ifndef PDQ_HOST_EMU
template <int N, int D>
__global__ void __launch_bounds__(64) lane_sample_kernel(SampleArgs a) {
  const size_t total = (size_t)a.n_inst * a.n_samples;
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (size_t g = (size_t)blockIdx.x * blockDim.x + threadIdx.x; g < total; g += stride) lane_sample<N, D>(a, g);
}
#endif

}  // namespace pdq
