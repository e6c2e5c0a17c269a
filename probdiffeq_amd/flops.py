"""Algorithmic FLOP model of the solver path (the reference's formulation).

Counts follow the operations the reference performs per call (LAPACK
R-only Householder QR(m, k) = 2 m k^2 - 2/3 k^3 for m >= k, GEMM 2abc,
triangular solve k^2 r, selector products H L counted as dense GEMMs), so
that ``achieved TFLOP/s = model FLOPs / measured kernel time`` compares
the kernels with the chip's FP64 peak on the work the algorithm requires,
not on what an implementation chooses to execute.

nc = covariance dimension (dense (nu+1) d, isotropic and per block nu+1),
mc = mean columns (dense 1, isotropic d, blockdiag 1), ko = observation
rows (dense d, isotropic 1, blockdiag 1 per block), nb = blocks (blockdiag
d, otherwise 1).
"""

from __future__ import annotations


def qr(m: int, k: int) -> float:
    """R-only Householder QR of an m x k matrix (LAPACK dgeqr2 count)."""
    if m < k:
        m, k = k, m
    return 2.0 * m * k * k - 2.0 / 3.0 * k**3


def gemm(a: int, b: int, c: int) -> float:
    return 2.0 * a * b * c


def trsm(k: int, r: int) -> float:
    return float(k * k * r)


def dims(cfg, n_tan: int = 0):
    """(nc, mc, ko, nb); with n_tan forward-mode directions every mean column carries n_tan
    tangent columns beside it (mc grows by the factor 1 + n_tan, the factors do not)."""
    N, d = cfg.num_derivatives + 1, cfg.ode_dim
    if cfg.factorisation == "dense":
        return N * d, 1 + n_tan, d, 1
    if cfg.factorisation == "isotropic":
        return N, d * (1 + n_tan), 1, 1
    return N, 1 + n_tan, 1, d


def _marginalise(nc, mc, rows_out):
    # (A chol)^T, QR of the stack, A mean
    return gemm(rows_out, nc, nc) + qr(nc + rows_out, rows_out) + gemm(rows_out, nc, mc)


def _revert(nc, mc, k):
    # (A chol)^T, QR of the (k + nc) block, gain solve, A mean, gain @ mean_observed
    return gemm(k, nc, nc) + qr(k + nc, k + nc) + trsm(k, nc) + gemm(k, nc, mc) + gemm(nc, k, mc)


def _merge(nc, mc):
    return gemm(nc, nc, nc) + gemm(nc, nc, mc) + gemm(nc, nc, nc) + qr(2 * nc, nc)


def attempt(cfg, n_tan: int = 0) -> float:
    """FLOPs of one attempted step (solver step + residual error estimate)."""
    nc, mc, ko, nb = dims(cfg, n_tan)
    f = 0.0
    lin = _marginalise(nc, mc, ko) + trsm(ko, mc)  # fx.marginalise(u) + whitened residual
    if cfg.constraint == "ts1":
        lin += gemm(ko, nc, 1)  # b = r(xi) - J xi
    if cfg.solver == "dynamic":
        f += gemm(nc, nc, mc)  # apply_flat (sigma = 1)
        f += lin
    if cfg.strategy == "filter":
        f += _marginalise(nc, mc, nc)
    else:
        f += _revert(nc, mc, nc)
        if cfg.strategy == "fixedpoint":
            f += _merge(nc, mc)
    f += _revert(nc, mc, ko)  # the update
    if cfg.solver != "dynamic":
        f += gemm(nc, nc, mc) + lin  # error estimate re-extrapolates and marginalises
    return nb * f


def interpolation(cfg) -> float:
    """FLOPs of one checkpoint interpolation beyond t1 (interpolate_fwd)."""
    nc, mc, _, nb = dims(cfg)
    if cfg.strategy == "filter":
        return nb * _marginalise(nc, mc, nc)
    f = 2 * _revert(nc, mc, nc)
    if cfg.strategy == "fixedpoint":
        f += _merge(nc, mc)
    return nb * f


def finalize_per_checkpoint(cfg) -> float:
    """Smoother backward pass: one conditional marginalisation per checkpoint."""
    nc, mc, _, nb = dims(cfg)
    if cfg.strategy == "filter":
        return 0.0
    return nb * _marginalise(nc, mc, nc)


def solve(cfg, attempts: float, checkpoints: int) -> float:
    """FLOPs of one solve with the given attempt count and number of checkpoints (K - 1)."""
    return attempts * attempt(cfg) + checkpoints * (interpolation(cfg) + finalize_per_checkpoint(cfg))


def lml_forward(cfg, grid_steps: int, observations: int, n_tan: int = 0) -> float:
    """Forward solve on the grid plus evaluate_lml's reverse scan; with n_tan > 0 the mean
    recursions carry the tangent columns of a forward-mode gradient (the factors are shared)."""
    nc, mc, ko, nb = dims(cfg, n_tan)
    step = attempt(cfg, n_tan) - (gemm(nc, nc, mc) + _marginalise(nc, mc, ko) + trsm(ko, mc))  # no error estimate
    lml = observations * (_marginalise(nc, mc, nc) + _revert(nc, mc, ko) + qr(ko, ko) + trsm(ko, mc))
    return nb * (grid_steps * step) + nb * lml


def lml_batch(cfg, n_inst: int, grid_steps: int, observations: int, n_tan: int = 0, reverse: bool = False) -> float:
    """FLOPs of a batch of isotropic lane LMLs without calibration (PDQ_SOLVER): the grid steps' factors
    once for the batch, and per instance the mean columns through them and the reverse scan (whose
    factors depend on the observation stds).  Per step and column: the transition N^2 + 3 N, the revert's
    and the merge's matrix-vector products 2 N^2 + 2 N each, the update 2 N + 1.  The reverse adjoint
    recomputes the means once and its step costs what a step of the means does."""
    N, d = cfg.num_derivatives + 1, cfg.ode_dim
    factors = lml_forward(cfg, grid_steps, 0, 0)
    column = 5 * N * N + 9 * N + 1
    per_inst = lml_forward(cfg, 0, observations, n_tan) + grid_steps * column * d * (1 + n_tan)
    if reverse:
        per_inst = 2 * lml_forward(cfg, 0, observations, 0) + 3 * grid_steps * column * d
    return factors + n_inst * per_inst


def lml_batch_bytes(cfg, n_inst: int, observations: int, grid_points: int, n_tan: int = 0, reverse: bool = False) -> float:
    """Algorithmic HBM bytes of the same: inputs and outputs (the Taylor coefficients carry their
    sensitivities), the shared records written and read once, and per instance the intervals' noise
    means (with their tangents), and for the adjoint node data, the means' adjoints and a checkpoint of
    the mean every 16 (nu = 3) or 12 (nu = 4) steps, each written and read once."""
    N, d = cfg.num_derivatives + 1, cfg.ode_dim
    n_theta = cfg.n_params + d
    shared = (grid_points - 1) * (4 * N + 2 * N * N + 1 + N * (N + 1)) + (observations - 1) * (N * N + N * (N + 1) // 2 + 2 * N)
    per_inst = (observations - 1) * N * d * (1 + n_tan)
    if reverse:
        per_inst = 2 * (observations - 1) * N * d + observations * (N + 1 + d) + (grid_points - 1) / (16 if N == 4 else 12) * N * d
    inputs = n_inst * (cfg.n_params + d + observations * (d + 1) + N * d * (1 + n_theta)) + grid_points
    return 8.0 * (inputs + n_inst * (1 + n_theta) + 2 * shared + 2 * n_inst * per_inst)


def solve_bytes(cfg, n_inst: int, K: int) -> float:
    """Algorithmic HBM bytes of one batched save_at solve: inputs, outputs written
    once, and the stored backward conditionals read back by the smoother's backward pass."""
    nc, mc, _, nb = dims(cfg)
    N, d = cfg.num_derivatives + 1, cfg.ode_dim
    ms = N * d                       # mean entries
    cs = nb * nc * nc                # factor entries
    inputs = cfg.n_params + N * d + K
    per_ckpt = 1 + ms + cs + nb + 1  # t, mean, chol, output_scale, num_steps
    reread = 0
    if cfg.strategy != "filter":
        cond = nb * nc * nc + ms + cs + 2 * nb * nc  # A, noise mean, noise chol, to_latent, to_observed
        per_ckpt += ms + cs + cond                   # filtering marginal + backward conditional
        reread = (K - 1) * cond
    return 8.0 * n_inst * (inputs + K * per_ckpt + reread)


def offgrid(cfg) -> float:
    """FLOPs of one off-grid marginal (solvers.py:149-203): the filter marginalises the transition;
    the fixed-interval smoother reverts it twice and marginalises one backward conditional."""
    nc, mc, _, nb = dims(cfg)
    if cfg.strategy == "filter":
        return nb * _marginalise(nc, mc, nc)
    return nb * (2 * _revert(nc, mc, nc) + _marginalise(nc, mc, nc))


def offgrid_bytes(cfg, n_query: int) -> float:
    """Algorithmic HBM bytes per batch of off-grid queries: each query reads its time, the two
    bracketing marginals (the filter needs one) and an output scale, and writes one marginal.  The
    binary search over the grid is not counted (it hits the cache)."""
    nc, mc, _, nb = dims(cfg)
    normal = nc * mc + nb * nc * nc
    reads = 1 + 1 + normal * (1 if cfg.strategy == "filter" else 2)
    return 8.0 * n_query * (reads + normal)
