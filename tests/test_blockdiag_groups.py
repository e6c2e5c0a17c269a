"""A block-diagonal workgroup of several wavefronts solves one instance after another in the same LDS
(pdq_bd.h).  On the CPU a group runs as threads with real barriers; here the lanes of its later
wavefronts leave every barrier late, so that the first one runs as far ahead as the barriers let it.
Whatever it writes for the next instance must not reach the last reads of this one.
"""

import numpy as np
import pytest


@pytest.fixture(scope="module")
def emu():
    from emu import emu as M

    M.build()
    M._lib = None
    return M


@pytest.mark.parametrize("strategy,solver,K", [("filter", "solver", 2), ("filter", "dynamic", 4), ("fixedinterval", "mle", 2)])
def test_the_next_instance_waits_for_the_last_reads(emu, strategy, solver, K):
    from probdiffeq_amd import capi

    d, nu, B = 66, 1, 3
    rng = np.random.default_rng(K)
    y0 = rng.normal(size=(B, d))
    dx = 1.0 / d
    f = -y0 * (np.roll(y0, -1, 1) - np.roll(y0, 1, 1)) / (2 * dx) + 0.05 * (np.roll(y0, -1, 1) - 2 * y0 + np.roll(y0, 1, 1)) / dx**2
    tc = np.stack([y0, f], axis=1).reshape(B, -1)
    p, t = np.tile([0.05, dx], (B, 1)), np.tile(np.linspace(0.0, 1e-4, K), (B, 1))
    cfg = capi.Config(factorisation="blockdiag", num_derivatives=nu, ode_dim=d, vector_field="burgers", n_params=2, strategy=strategy, solver=solver)
    alone = [emu.solve(cfg, p[i : i + 1], tc[i : i + 1], t[i : i + 1], fixed_grid=True) for i in range(B)]
    emu.lib().pdqemu_set_lag(64, 20000)
    try:
        together = emu.solve(cfg, p, tc, t, fixed_grid=True)
    finally:
        emu.lib().pdqemu_set_lag(0, 0)
    for key, x in together.items():
        assert np.array_equal(x, np.concatenate([a[key] for a in alone]), equal_nan=True), key
