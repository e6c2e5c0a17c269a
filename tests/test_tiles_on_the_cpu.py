"""The kernels that pass data between lanes through LDS (pdq_lane_sample.h, pdq_lane_offgrid.h,
pdq_lane_lml_shared.h) on the CPU: whole workgroups as threads with real barriers, one per wavefront
and one per workgroup.  The references are NumPy's recursion, a query alone, and the LML's code that
computes every instance's own factors.
"""

import numpy as np
import pytest


@pytest.fixture(scope="module")
def emu():
    from emu import emu as M

    M.build()
    M._lib = None
    return M


@pytest.mark.parametrize(  # (the conditionals are read together from 16 samples on)
    "nu,B,K,S,staged",
    [(3, 1, 2, 1, False), (4, 3, 7, 21, False), (3, 2, 8, 40, False), (4, 2, 5, 3, False), (4, 3, 7, 21, True), (3, 2, 8, 40, True),
     (4, 5, 6, 16, True), (3, 5, 9, 27, True)],
)
def test_samples(emu, nu, B, K, S, staged):
    from probdiffeq_amd import capi

    N, d = nu + 1, 2
    rng = np.random.default_rng(K)
    r = lambda *shape: rng.normal(size=shape)
    sol = dict(cond_A=0.3 * r(B, K - 1, N, N), cond_mean=r(B, K - 1, N, d), cond_chol=np.tril(r(B, K - 1, N, N)), cond_tl=r(B, K - 1, N),
               cond_to=r(B, K - 1, N), term_mean=r(B, N, d), term_chol=np.tril(r(B, N, N)))
    base = r(B, S, K, N)
    cfg = capi.Config(factorisation="isotropic", num_derivatives=nu, strategy="fixedinterval", solver="dynamic")
    got = emu.sample(cfg, sol, base, staged=staged).reshape(B, S, K, N, d)
    x = sol["term_mean"][:, None] + np.einsum("bij,bsj->bsi", sol["term_chol"], base[:, :, K - 1])[..., None]
    for k in range(K - 1, -1, -1):
        if k < K - 1:
            A = sol["cond_to"][:, k, :, None] * sol["cond_A"][:, k]
            L = np.abs(sol["cond_to"][:, k, :, None]) * sol["cond_chol"][:, k]
            x = A[:, None] @ (sol["cond_tl"][:, k, :, None][:, None] * x) + sol["cond_mean"][:, k][:, None] + L[:, None] @ base[:, :, k][..., None]
        # 2 N + 6 operations per point, K points, entries up to 1e3 times the result's
        assert np.abs(got[:, :, k] - x).max() <= (2 * N + 6) * K * 2.0**-53 * 1e3 * np.abs(x).max(), k


@pytest.mark.parametrize("strategy", ["filter", "fixedinterval"])
@pytest.mark.parametrize("nu,B,K,M", [(3, 3, 2, 1), (4, 2, 7, 63), (3, 1, 9, 65), (4, 30, 5, 5), (3, 1, 1601, 70)])
def test_offgrid_queries(emu, nu, B, K, M, strategy):
    """A query's result is the same bits alone and among others, in one wavefront or across two."""
    from probdiffeq_amd import capi

    N, d = nu + 1, 2
    rng = np.random.default_rng(K)
    t = np.cumsum(rng.uniform(0.1, 0.3, (B, K)), axis=1)
    j, w = rng.integers(1, K, (B, M)), rng.uniform(0.1, 0.9, (B, M))
    tq = np.take_along_axis(t, j - 1, 1) * w + np.take_along_axis(t, j, 1) * (1 - w)
    chol = lambda: (np.tril(rng.normal(size=(B, K, N, N))) + 3 * np.eye(N)).reshape(B, K, -1)
    sol = {"mean": rng.normal(size=(B, K, N * d)), "chol": chol(), "output_scale": rng.uniform(0.5, 2.0, (B, K, 1))}
    if strategy != "filter":
        sol |= {"filt_mean": rng.normal(size=(B, K, N * d)), "filt_chol": chol()}
    cfg = capi.Config(factorisation="isotropic", num_derivatives=nu, strategy=strategy, solver="dynamic")
    together = emu.offgrid(cfg, t, sol, tq)
    for b in range(min(B, 2)):
        for q in {0, M // 2, M - 1}:
            alone = emu.offgrid(cfg, t[b : b + 1], {k: v[b : b + 1] for k, v in sol.items()}, tq[b : b + 1, q : q + 1])
            for x, y in zip(together, alone):
                assert np.array_equal(x[b, q], y[0, 0])


def _lml_inputs(B, steps, every):
    rng = np.random.default_rng(steps)
    P = np.tile([0.5, 0.05, 0.5, 0.05], (B, 1)) * rng.uniform(0.8, 1.2, (B, 4))
    Y = rng.uniform(4.0, 20.0, (B, 2))
    grid = np.cumsum(np.concatenate([[0.1], rng.uniform(0.005, 0.02, steps)]))
    data = Y[:, None] * rng.uniform(0.9, 1.1, (B, steps // every + 1, 2))
    return P, Y, grid, every, data, rng.uniform(0.1, 0.5, (B, steps // every + 1))


@pytest.mark.parametrize(
    "nu,B,steps,every,late",
    [(3, 1, 1, 1, None), (4, 2, 3, 3, None), (3, 11, 17, 1, None), (4, 2, 64, 16, None), (3, 2, 65, 5, None), (4, 1, 25, 5, (0, 64)),
     (3, 1, 49, 7, (64, 128)), (3, 2, 385, 1, None), (4, 1, 392, 7, None)],
)
def test_lml_with_the_factors_once(emu, nu, B, steps, every, late):
    """Value, tangents and adjoint; `late`: one of the adjoint's two wavefronts leaves every barrier
    late.  About 100 operations in another order per step, amplified a hundredfold: 1.1e-12 per step."""
    from probdiffeq_amd import capi

    args = _lml_inputs(B, steps, every)
    cfg = capi.Config(factorisation="isotropic", num_derivatives=nu, strategy="fixedpoint", solver="solver")
    v0, g0 = emu.lml(cfg, *args, kernel="lane")
    runs = []
    if late:
        emu.lib().pdqemu_set_lag(*late, 3000)
    try:
        runs.append(emu.lml_shared(cfg, *args, reverse=True))
    finally:
        emu.lib().pdqemu_set_lag(0, 0, 0)
    runs.append(emu.lml_shared(cfg, *args))
    value = emu.lml_shared(cfg, *args, grad=False)[0]
    assert np.array_equal(value, runs[1][0])  # with a gradient and without: the same bits
    tol = 1.1e-12 * max(steps, 130)
    for v, g in runs:
        assert np.abs(v - v0).max() <= tol * np.abs(v0).max()
        assert np.abs(g - g0).max() <= tol * np.abs(g0).max()
