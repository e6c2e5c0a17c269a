"""The fixed-shape cooperative kernels (pdq_coop_wave.h) with their options, bit for bit against the
run-time-shape kernel at 64 lanes per instance: clipped steps, the proportional-integral controller,
the other error norm, the error per unit step, and the solvers without dynamic calibration.  The option
error_re_linearize, which only the run-time-shape kernel holds, changes nothing here: solver_dynamic
calibrates at the point it would linearise at again, and a dense prediction's mean is the
extrapolation's, from the same products.
"""

import numpy as np
import pytest

import test_gpu_parity as T

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

OPTIONS = [dict(clip_dt=True), dict(control="proportional_integral"), dict(error_norm="rms_then_scale"), dict(error_per_unit_step=True),
           dict(clip_dt=True, control="proportional_integral", error_norm="rms_then_scale", init_std=0.1, base_output_scale=2.0)]


@pytest.mark.parametrize("kw", OPTIONS, ids=lambda kw: "-".join(kw))
@pytest.mark.parametrize(
    "fact,nu,strategy,solver,constraint",
    [("dense", 2, "fixedpoint", "dynamic", "ts1"), ("dense", 4, "filter", "dynamic", "ts0"), ("dense", 5, "fixedinterval", "dynamic", "ts0"),
     ("isotropic", 2, "filter", "dynamic", "ts1"), ("isotropic", 5, "fixedpoint", "dynamic", "ts0"), ("dense", 3, "filter", "solver", "ts0"),
     ("dense", 4, "fixedinterval", "mle", "ts0"), ("dense", 2, "filter", "mle", "ts1")],
)
def test_options_equal_the_run_time_shape_kernel(fact, nu, strategy, solver, constraint, kw):
    from probdiffeq_amd import capi

    capi.require_device()
    print(f"wave option case: {fact} nu={nu} {strategy} {solver} {constraint} {kw}", flush=True)
    p, y, t = T._lv_batch(9, seed=nu, t_lo=2.0, t_hi=6.0, K=6)
    P, Y, S = T._dev(p), T._dev(y), T._dev(t)
    tc = capi.taylor_coefficients("lotka_volterra", P, Y, 0.0, nu)
    runs = []
    for option in (False, True):
        cfg = capi.Config(factorisation=fact, num_derivatives=nu, strategy=strategy, solver=solver, constraint=constraint, rtol=1e-4, atol=1e-6,
                          lanes_per_instance=64, error_re_linearize=option, **kw)
        runs.append(capi.solve(cfg, P, tc, S))
    assert int(runs[0]["status"].abs().sum()) == 0
    for key in runs[0]:
        a, b = (r[key].cpu().numpy() for r in runs)
        assert np.array_equal(a, b, equal_nan=a.dtype.kind == "f"), key
