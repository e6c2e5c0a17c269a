"""A block-diagonal workgroup of several wavefronts solves one instance after another in the same LDS
(pdq_bd.h).  On the CPU a group runs as threads with real barriers; here the lanes of its later
wavefronts leave every barrier late, so that the first one runs as far ahead as the barriers let it.
Whatever it writes for the next instance must not reach the last reads of this one.
"""

import numpy as np
import pytest

import test_gpu_parity as T

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def emu():
    from emu import emu as M

    M.build()
    M._lib = None
    return M


@pytest.mark.parametrize(
    "strategy,solver,K,grid",
    [("filter", "solver", 2, True), ("filter", "dynamic", 4, True), ("fixedinterval", "mle", 2, True),
     ("filter", "dynamic", 2, False), ("fixedpoint", "dynamic", 2, False), ("fixedinterval", "solver", 2, False)],
)
def test_the_next_instance_waits_for_the_last_reads(emu, strategy, solver, K, grid):
    from probdiffeq_amd import capi

    d, nu, B = 66, 1, 3
    rng = np.random.default_rng(K)
    y0 = rng.normal(size=(B, d))
    dx = 1.0 / d
    f = -y0 * (np.roll(y0, -1, 1) - np.roll(y0, 1, 1)) / (2 * dx) + 0.05 * (np.roll(y0, -1, 1) - 2 * y0 + np.roll(y0, 1, 1)) / dx**2
    tc = np.stack([y0, f], axis=1).reshape(B, -1)
    p, t = np.tile([0.05, dx], (B, 1)), np.tile(np.linspace(0.0, 1e-4, K), (B, 1))
    cfg = capi.Config(factorisation="blockdiag", num_derivatives=nu, ode_dim=d, vector_field="burgers", n_params=2, strategy=strategy, solver=solver,
                      dt0=4e-5, rtol=1e-3, atol=1e-4)
    alone = [emu.solve(cfg, p[i : i + 1], tc[i : i + 1], t[i : i + 1], fixed_grid=grid) for i in range(B)]
    emu.lib().pdqemu_set_lag(64, 128, 20000)
    try:
        together = emu.solve(cfg, p, tc, t, fixed_grid=grid)
        print(together["attempts"])
    finally:
        emu.lib().pdqemu_set_lag(0, 0, 0)
    for key, x in together.items():
        assert np.array_equal(x, np.concatenate([a[key] for a in alone]), equal_nan=True), key


@pytest.mark.gpu
@pytest.mark.parametrize("d", [2, 33, 65, 130])
@pytest.mark.parametrize("nu", [4, 5])
@pytest.mark.parametrize("strategy", ["fixedpoint", "fixedinterval"])
def test_high_order_smoothers(oracle, strategy, nu, d):
    """The kernels with the most scratch memory per lane: against the oracle, and the same bits again."""
    from probdiffeq_amd import capi

    capi.require_device()
    print(f"blockdiag smoother case: {strategy} nu={nu} d={d}", flush=True)
    rng = np.random.default_rng(d)
    B = 3
    params, y0, times = np.full((B, 1), 1.5), rng.uniform(0.1, 0.9, size=(B, d)), np.tile(np.linspace(0.0, 3.0, 5), (B, 1))
    cfg = capi.Config(factorisation="blockdiag", num_derivatives=nu, ode_dim=d, vector_field="logistic", n_params=1, strategy=strategy,
                      rtol=1e-5, atol=1e-7)
    T._compare(oracle, capi, cfg, params, y0, times)
    P, S = T._dev(params), T._dev(times)
    tc = capi.taylor_coefficients("logistic", P, T._dev(y0), 0.0, nu)
    once = {k: v.cpu().numpy() for k, v in capi.solve(cfg, P, tc, S).items() if v is not None}
    for _ in range(3):
        for key, x in capi.solve(cfg, P, tc, S).items():
            if x is not None:
                assert np.array_equal(x.cpu().numpy(), once[key], equal_nan=once[key].dtype.kind == "f"), key


@pytest.mark.gpu
@pytest.mark.parametrize("strategy", ["filter", "fixedinterval"])
def test_more_instances_than_workgroups_on_a_fixed_grid(strategy):
    """Workgroups that take several instances on a fixed grid (an odd number of steps): an instance's
    result is the same bits as alone."""
    from probdiffeq_amd import capi

    capi.require_device()
    print(f"blockdiag fixed grid case: {strategy}", flush=True)
    d, nu, B = 130, 2, 3000
    rng = np.random.default_rng(7)
    y0 = rng.normal(size=(B, d))
    cfg = capi.Config(factorisation="blockdiag", num_derivatives=nu, ode_dim=d, vector_field="burgers", n_params=2, strategy=strategy)
    P, Y, S = T._dev(np.tile([0.05, 1.0 / d], (B, 1))), T._dev(y0), T._dev(np.tile(np.linspace(0.0, 1e-4, 4), (B, 1)))
    tc = capi.taylor_coefficients("burgers", P, Y, 0.0, nu)
    run = lambda rows: capi.solve(cfg, P[rows], tc[rows], S[rows], fixed_grid=True)
    together = run(slice(None))
    for rows in (slice(0, 64), slice(B - 64, B)):
        alone = run(rows)
        for key in ("mean", "chol"):
            assert torch.equal(together[key][rows], alone[key]), (key, rows)
