"""The block-diagonal filter's kernels for the default options (pdq_bd.h) against the kernels for
every option, bit for bit: with solver_dynamic the option error_re_linearize changes nothing in the
results (the calibration linearises at the same point), but only the latter hold it.  The sizes are
the edges of the lane groups: powers of two within a wavefront, and one wavefront more than fits.
"""

import numpy as np
import pytest

import test_gpu_parity as T

torch = pytest.importorskip("torch")


@pytest.mark.gpu
@pytest.mark.parametrize("control", ["integral", "proportional_integral"])
@pytest.mark.parametrize("nu,d", [(1, 16), (2, 3), (2, 8), (2, 33), (2, 64), (2, 65), (2, 512), (3, 17), (3, 130), (4, 129), (5, 70)])
def test_default_option_kernel_equals_the_kernel_for_every_option(nu, d, control):
    from probdiffeq_amd import capi

    capi.require_device()
    print(f"blockdiag case: nu={nu} d={d} {control}", flush=True)
    rng = np.random.default_rng(d)
    x = np.arange(d) / d
    y0 = np.stack([sum(rng.normal(0, 1 / k) * np.sin(2 * np.pi * k * x) for k in range(1, 4)) for _ in range(5)])
    P, Y = T._dev(np.tile([0.05, 1.0 / d], (5, 1))), T._dev(y0)
    S = T._dev(np.tile(np.linspace(0.0, 0.05, 4), (5, 1)))
    tc = capi.taylor_coefficients("burgers", P, Y, 0.0, nu)
    runs = []
    for option in (False, True):
        cfg = capi.Config(factorisation="blockdiag", num_derivatives=nu, ode_dim=d, vector_field="burgers", n_params=2, strategy="filter",
                          solver="dynamic", rtol=1e-4, atol=1e-6, control=control, error_re_linearize=option)
        runs.append(capi.solve(cfg, P, tc, S))
    for key in runs[0]:
        if runs[0][key] is None:
            continue
        a, b = (r[key].cpu().numpy() for r in runs)
        assert np.array_equal(a, b, equal_nan=a.dtype.kind == "f"), key
