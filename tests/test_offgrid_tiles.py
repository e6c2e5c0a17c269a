"""The off-grid kernel's wavefront tiles (pdq_lane_offgrid.h): 64 consecutive queries gather their
grid points' rows and write their results together.  A query's result has to be the same bits
whatever its neighbours are: in wavefronts of one instance (grid searched in LDS), of several, partly
filled, and on grids too long for the LDS search.  tests/test_gpu_offgrid.py holds the values to the
oracle.
"""

import numpy as np
import pytest

import test_gpu_parity as T

torch = pytest.importorskip("torch")


@pytest.mark.gpu
@pytest.mark.parametrize("strategy", ["filter", "fixedinterval"])
@pytest.mark.parametrize("nu,B,K,M", [(3, 5, 2, 1), (4, 3, 7, 63), (3, 2, 40, 64), (4, 4, 9, 65), (3, 70, 5, 3), (4, 2, 2241, 130), (3, 2, 1601, 70)])
def test_results_do_not_depend_on_the_neighbours(nu, B, K, M, strategy):
    from probdiffeq_amd import capi

    capi.require_device()
    print(f"offgrid tile case: nu={nu} B={B} K={K} M={M} {strategy}", flush=True)
    N, d = nu + 1, 2
    rng = np.random.default_rng(K)
    t = np.cumsum(rng.uniform(0.1, 0.3, (B, K)), axis=1)
    j = rng.integers(1, K, (B, M))
    w = rng.uniform(0.1, 0.9, (B, M))
    tq = np.take_along_axis(t, j - 1, 1) * w + np.take_along_axis(t, j, 1) * (1 - w)
    chol = lambda: (np.tril(rng.normal(size=(B, K, N, N))) + 3 * np.eye(N)).reshape(B, K, -1)
    sol = {"mean": rng.normal(size=(B, K, N * d)), "chol": chol(), "filt_mean": rng.normal(size=(B, K, N * d)), "filt_chol": chol(),
           "output_scale": rng.uniform(0.5, 2.0, (B, K, 1))}
    cfg = capi.Config(factorisation="isotropic", num_derivatives=nu, strategy=strategy, solver="dynamic")

    def run(rows, cols):
        out = {k: T._dev(v[rows]) for k, v in sol.items()}
        return [x.cpu().numpy() for x in capi.offgrid_marginals(cfg, out, T._dev(t[rows]), T._dev(tq[rows][:, cols]))]

    together = run(slice(None), slice(None))
    for b in range(min(B, 4)):
        for cols in (slice(None), slice(M // 2, M // 2 + 1)):
            alone = run(slice(b, b + 1), cols)
            for x, y in zip(together, alone):
                assert np.array_equal(x[b, cols], y[0])
