"""The LML with the batch's factors computed once at the edges of its launches
(pdq_lane_lml_shared_launch.h): the shortest grids (up to 64 steps the factors are one launch), and the
grids from which it runs in chunks (384 steps: six chunks of 64; a last chunk of one step, of one interval).  Value
and forward gradient against the cooperative kernel, the reverse adjoint against the forward
gradient.  The tolerance allows for about 100 operations in another order per step (1.1e-14) amplified
a hundredfold, over at least 130 steps: 1.5e-10.
"""

import numpy as np
import pytest

import test_gpu_parity as T

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _inputs(B, steps, every):
    rng = np.random.default_rng(steps)
    P = np.tile([0.5, 0.05, 0.5, 0.05], (B, 1)) * rng.uniform(0.8, 1.2, (B, 4))
    Y = rng.uniform(4.0, 20.0, (B, 2))
    grid = np.cumsum(np.concatenate([[0.1], rng.uniform(0.005, 0.02, steps)]))
    data = Y[:, None] * rng.uniform(0.9, 1.1, (B, steps // every + 1, 2))
    stds = rng.uniform(0.1, 0.5, (B, steps // every + 1))
    return [T._dev(x) for x in (P, Y, grid)], (T._dev(data), T._dev(stds))


def _run(nu, args, every, obs, grad=True, **kw):
    from probdiffeq_amd import capi

    cfg = capi.Config(factorisation="isotropic", num_derivatives=nu, strategy="fixedpoint", **{"solver": "solver", **kw})
    v, g = capi.lml_value_and_grad(cfg, *args, every, *obs, grad=grad)
    return v.cpu().numpy(), g.cpu().numpy() if grad else None


def _close(a, b, steps):
    tol = 1.1e-12 * max(steps, 130)
    assert np.abs(a[0] - b[0]).max() <= tol * np.abs(b[0]).max()
    if a[1] is not None and b[1] is not None:
        assert (np.abs(a[1] - b[1]).max(0) <= tol * np.abs(b[1]).max()).all()


@pytest.mark.parametrize(
    "nu,B,steps,every",
    [(3, 1, 1, 1), (3, 65, 2, 1), (3, 3, 3, 3), (3, 65, 4, 2), (3, 2, 7, 7), (3, 65, 8, 8), (3, 1, 11, 11), (3, 65, 12, 4), (3, 2731, 8, 4), (3, 66, 64, 1),
     (4, 1, 1, 1), (4, 65, 1, 1), (4, 63, 2, 2), (4, 2, 3, 1), (4, 65, 7, 7), (4, 1, 8, 8), (4, 64, 9, 3), (4, 3, 64, 32), (4, 2, 65, 13),
     (3, 66, 384, 8), (3, 2, 385, 1), (4, 65, 392, 7), (4, 3, 448, 64), (3, 5, 320, 5)],
)
def test_edges_of_the_dispatch(nu, B, steps, every):
    print(f"lml short case: nu={nu} B={B} steps={steps} every={every}", flush=True)
    args, obs = _inputs(B, steps, every)
    forward = _run(nu, args, every, obs)
    _close(_run(nu, args, every, obs, lanes_per_instance=16), forward, steps)
    _close(_run(nu, args, every, obs, lml_gradient="reverse"), forward, steps)
    _close(_run(nu, args, every, obs, grad=False), forward, steps)


@pytest.mark.parametrize("nu,steps,every", [(3, 40, 10), (4, 30, 3), (4, 1, 1)])
def test_calibrated_adjoint_on_a_partial_segment(nu, steps, every):
    """solver_dynamic keeps the lane kernels: its adjoint with one segment of fewer than 50 steps."""
    print(f"lml dynamic case: nu={nu} steps={steps} every={every}", flush=True)
    args, obs = _inputs(65, steps, every)
    forward = _run(nu, args, every, obs, solver="dynamic")
    _close(_run(nu, args, every, obs, solver="dynamic", lml_gradient="reverse"), forward, steps)
