"""The fixed-shape cooperative kernels (pdq_coop_wave.h): one instance per wavefront, the QR in
registers.

On the CPU their code runs as 64 threads per instance with real barriers (a missed one would
deadlock) against the oracle.  On the GPU they have to reproduce the run-time-shape kernel at 64 lanes
per instance bit for bit (the coarse fixed grids diverge for some instances, infinities and NaN
included): with solver_dynamic the option error_re_linearize changes nothing in the
results (the calibration linearises at the same point), but only the run-time-shape kernel holds it.
"""

import numpy as np
import pytest

import test_gpu_parity as T
import test_kernel_emulation as E

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def emu():
    from emu import emu as M

    M.build()
    M._lib = None
    return M


@pytest.mark.parametrize(
    "fact,nu,strategy,solver,constraint,fixed_grid",
    [
        ("dense", 2, "filter", "dynamic", "ts0", False),
        ("dense", 4, "filter", "solver", "ts1", False),
        ("dense", 3, "fixedpoint", "dynamic", "ts1", False),
        ("dense", 2, "fixedinterval", "mle", "ts0", False),
        ("dense", 5, "fixedinterval", "dynamic", "ts0", True),
        ("isotropic", 2, "fixedpoint", "mle", "ts1", False),
        ("isotropic", 5, "filter", "dynamic", "ts0", False),
    ],
)
def test_wave_code_against_the_oracle(oracle, emu, fact, nu, strategy, solver, constraint, fixed_grid):
    from probdiffeq_amd import capi

    cfg = capi.Config(factorisation=fact, num_derivatives=nu, strategy=strategy, solver=solver, constraint=constraint, rtol=1e-3, atol=1e-5)
    p, y, t = T._lv_batch(1, seed=7, t_lo=1.0, t_hi=1.5, K=4)
    E._run(oracle, emu, cfg, p, y, t, fixed_grid=fixed_grid, kernel="wave")


def _matern(nu, length_scale=0.4):
    """The drift of a Matern prior (ssm_impl_api.py:443-477): its 1-norm makes larger steps double."""
    import math

    N, z = nu + 1, math.sqrt(2 * (nu + 0.5)) / length_scale
    return np.concatenate([-math.comb(N, i) * z ** (N - i) * np.eye(2) for i in range(N)], axis=1)


@pytest.mark.parametrize("nu,solver", [(2, "dynamic"), (3, "solver")])
def test_wave_code_with_an_exponential_prior(oracle, emu, nu, solver):
    from probdiffeq_amd import capi

    cfg = capi.Config(factorisation="dense", num_derivatives=nu, strategy="filter", solver=solver, rtol=1e-3, atol=1e-5,
                      prior="exponential", prior_drift=_matern(nu))
    p, y, t = T._lv_batch(1, seed=7, t_lo=0.6, t_hi=0.9, K=3)
    E._run(oracle, emu, cfg, p, y, t, kernel="wave")


@pytest.mark.gpu
@pytest.mark.parametrize("constraint", ["ts0", "ts1"])
@pytest.mark.parametrize("nu", [2, 3, 4, 5])
def test_wave_kernel_with_an_exponential_prior_equals_the_run_time_shape_kernel(nu, constraint):
    from probdiffeq_amd import capi

    capi.require_device()
    print(f"wave case: matern nu={nu} {constraint}", flush=True)
    p, y, t = T._lv_batch(17, seed=nu, t_lo=1.0, t_hi=3.0, K=7)
    P, Y, S = T._dev(p), T._dev(y), T._dev(t)
    tc = capi.taylor_coefficients("lotka_volterra", P, Y, 0.0, nu)
    runs = []
    for option in (False, True):
        cfg = capi.Config(factorisation="dense", num_derivatives=nu, strategy="filter", solver="dynamic", constraint=constraint, rtol=1e-4,
                          atol=1e-6, lanes_per_instance=64, error_re_linearize=option, prior="exponential", prior_drift=T._dev(_matern(nu)))
        runs.append(capi.solve(cfg, P, tc, S))
    assert int(runs[0]["status"].abs().sum()) == 0
    for key in runs[0]:
        a, b = (r[key].cpu().numpy() for r in runs)
        assert np.array_equal(a, b, equal_nan=a.dtype.kind == "f"), key


@pytest.mark.gpu
@pytest.mark.parametrize("constraint", ["ts0", "ts1"])
@pytest.mark.parametrize("strategy", ["filter", "fixedpoint", "fixedinterval"])
@pytest.mark.parametrize("fact,nu", [("dense", 2), ("dense", 3), ("dense", 4), ("dense", 5), ("isotropic", 2), ("isotropic", 5)])
def test_wave_kernel_equals_the_run_time_shape_kernel(fact, nu, strategy, constraint):
    from probdiffeq_amd import capi

    capi.require_device()
    print(f"wave case: {fact} nu={nu} {strategy} {constraint}", flush=True)
    p, y, t = T._lv_batch(33, seed=nu, t_lo=2.0, t_hi=8.0, K=11)
    P, Y, S = T._dev(p), T._dev(y), T._dev(t)
    tc = capi.taylor_coefficients("lotka_volterra", P, Y, 0.0, nu)
    for grid in (False, True):
        runs = []
        for option in (False, True):
            cfg = capi.Config(factorisation=fact, num_derivatives=nu, strategy=strategy, solver="dynamic", constraint=constraint,
                              rtol=1e-5, atol=1e-7, lanes_per_instance=64, error_re_linearize=option)
            runs.append(capi.solve(cfg, P, tc, S, fixed_grid=grid))
        assert int(runs[0]["status"].abs().sum()) == 0
        for key in runs[0]:
            a, b = (r[key].cpu().numpy() for r in runs)
            assert np.array_equal(a, b, equal_nan=a.dtype.kind == "f"), (key, grid)
