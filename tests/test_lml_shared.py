"""The LML with the factors computed once for the batch (pdq_lane_lml_shared.h; isotropic, ts0,
solver): value and forward gradient against the cooperative kernel, which computes every instance's
own factors, and the reverse adjoint against the forward gradient.  The sizes are the edges of its
tiles: 16 steps staged at once, 64 steps' preconditioners, 64 lanes, intervals of one step and of the
whole grid.  The tolerance allows for the different order of about 100 operations in each of 130
steps (130 * 100 * 1.1e-16 = 1.5e-12) amplified a hundredfold.
"""

import numpy as np
import pytest

import test_gpu_parity as T

torch = pytest.importorskip("torch")

FIELDS = {"lotka_volterra": [0.5, 0.05, 0.5, 0.05], "van_der_pol": [1.5], "linear": [-0.5, 0.3], "logistic": [0.7], "burgers": [0.02, 0.5]}


@pytest.mark.gpu
@pytest.mark.parametrize(
    "nu,B,steps,every,field",
    [(3, 1, 8, 8, "lotka_volterra"), (4, 3, 15, 5, "van_der_pol"), (3, 65, 16, 1, "linear"), (4, 64, 17, 17, "logistic"), (3, 2, 63, 9, "burgers"),
     (4, 70, 64, 16, "lotka_volterra"), (3, 11, 65, 13, "lotka_volterra"), (4, 5, 130, 2, "linear"), (3, 33, 128, 64, "van_der_pol")],
)
def test_shared_factors(nu, B, steps, every, field):
    from probdiffeq_amd import capi

    capi.require_device()
    print(f"lml case: nu={nu} B={B} steps={steps} every={every} {field}", flush=True)
    rng = np.random.default_rng(steps)
    K = steps + 1
    P = np.tile(FIELDS[field], (B, 1)) * rng.uniform(0.8, 1.2, (B, len(FIELDS[field])))
    Y = rng.uniform(0.2, 1.0, (B, 2)) * (20.0 if field == "lotka_volterra" else 1.0)
    grid = np.cumsum(np.concatenate([[0.1], rng.uniform(0.005, 0.02, steps)]))
    Kobs = steps // every + 1
    data, stds = Y[:, None] * rng.uniform(0.9, 1.1, (B, Kobs, 2)), rng.uniform(0.1, 0.5, (B, Kobs))
    args = [T._dev(x) for x in (P, Y, grid)]

    def run(**kw):
        cfg = capi.Config(factorisation="isotropic", num_derivatives=nu, strategy="fixedpoint", solver="solver", vector_field=field,
                          n_params=P.shape[1], **kw)
        return [x.cpu().numpy() for x in capi.lml_value_and_grad(cfg, *args, every, T._dev(data), T._dev(stds))]

    value, grad = run()
    reverse = run(lml_gradient="reverse")
    own = run(lanes_per_instance=16)
    for v, g in (reverse, own):
        assert np.abs(v - value).max() <= 1.5e-10 * np.abs(value).max()
        assert (np.abs(g - grad).max(0) <= 1.5e-10 * np.abs(grad).max()).all()
