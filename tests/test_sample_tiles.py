"""The posterior sampler's wavefront tiles (pdq_lane_sample.h): four points at a time through LDS,
the conditionals loaded by each lane or, with 16 samples and more in a large batch, together.  Against
the same recursion in NumPy, within the rounding bound that runs along with it.  The sizes are the
edges: fewer points than a tile, every remainder, partly filled wavefronts, and 64-row windows that
meet one to five instances.
"""

import numpy as np
import pytest

import test_gpu_parity as T

torch = pytest.importorskip("torch")


@pytest.mark.gpu
@pytest.mark.parametrize(
    "nu,B,K,S",
    [(3, 1, 2, 1), (4, 3, 5, 5), (3, 7, 4, 3), (4, 5, 11, 15), (3, 2, 6, 40),  # every lane its own conditionals
     (4, 2049, 5, 16), (3, 2000, 8, 17), (4, 513, 7, 64), (3, 530, 6, 63), (4, 40, 9, 1000)],  # together
)
def test_samples_equal_the_recursion(nu, B, K, S):
    from probdiffeq_amd import capi

    capi.require_device()
    print(f"sample case: nu={nu} B={B} K={K} S={S}", flush=True)
    N, d, eps = nu + 1, 2, 2.0**-53
    rng = np.random.default_rng(K)
    r = lambda *shape: rng.normal(size=shape)
    sol = dict(cond_A=0.3 * r(B, K - 1, N, N), cond_mean=r(B, K - 1, N, d), cond_chol=np.tril(r(B, K - 1, N, N)), cond_tl=r(B, K - 1, N),
               cond_to=r(B, K - 1, N), term_mean=r(B, N, d), term_chol=np.tril(r(B, N, N)))
    base = r(B, S, K, N)
    cfg = capi.Config(factorisation="isotropic", num_derivatives=nu, strategy="fixedinterval", solver="dynamic")
    out = {k: T._dev(v.reshape(B, -1) if k.startswith("term") else v.reshape(B, K - 1, -1)) for k, v in sol.items()}
    got = capi.sample(cfg, out, K, T._dev(base)).cpu().numpy().reshape(B, S, K, N, d)
    rounding = (2 * N + 6) * eps  # of one point: products, sums and the scalings, on both sides
    lz = np.einsum("bij,bsj->bsi", sol["term_chol"], base[:, :, K - 1])[..., None]
    x = sol["term_mean"][:, None] + lz
    err = 2 * rounding * (np.abs(sol["term_mean"])[:, None] + np.einsum("bij,bsj->bsi", np.abs(sol["term_chol"]), np.abs(base[:, :, K - 1]))[..., None])
    assert (np.abs(got[:, :, K - 1] - x) <= err).all()
    for k in range(K - 2, -1, -1):
        A = sol["cond_to"][:, k, :, None] * sol["cond_A"][:, k]
        L = np.abs(sol["cond_to"][:, k, :, None]) * sol["cond_chol"][:, k]
        tl, m, z = sol["cond_tl"][:, k, :, None][:, None], sol["cond_mean"][:, k][:, None], base[:, :, k]
        mag = np.abs(A)[:, None] @ np.abs(tl * x) + np.abs(m) + (np.abs(L)[:, None] @ np.abs(z)[..., None])
        err = np.abs(A)[:, None] @ (np.abs(tl) * err) + 2 * rounding * mag
        x = A[:, None] @ (tl * x) + m + L[:, None] @ z[..., None]
        assert (np.abs(got[:, :, k] - x) <= err).all(), k
