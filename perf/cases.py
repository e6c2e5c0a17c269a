"""The workloads whose time and results are followed on one MI355X.

Each case is one call of a public entry point as a user's program makes it: a
single adaptive solve (the plain drop-in), batched adaptive solves in the three
factorisations, the marginal log-likelihood with its gradient in both modes,
off-grid marginals and posterior samples.  The inputs are synthetic draws of
the Lotka-Volterra, van der Pol and Burgers problems that bench.py and the
tests solve.

`exact` restates what a case returns in plain torch, float64: an adaptive
square-root filter / smoother on a whole batch at once, with its own Householder
factorisation and its own transition matrices.  Square-root factors are only
defined up to the signs of their columns, so `exact` gives the means, output
scales, times, log-likelihoods, gradients and samples, and None for factors and
for the counts of steps.  It gives no smoothed means of adaptive solves either:
where a step ends a rounding's breadth behind a save point (dt near eps), the
backward conditional across that gap is scaled by dt^-nu and 64 bits do not
determine what it maps to.
"""

import math
from fractions import Fraction

import numpy as np
import torch

from probdiffeq_amd import capi, ivpsolve, torch_ops
from probdiffeq_amd import probdiffeq as pdq

F64 = torch.float64
THETA0 = np.array([0.5, 0.05, 0.5, 0.05])
DT0, EPS, SAFETY, FACTOR_MIN, FACTOR_MAX = 0.1, 1e-8, 0.95, 0.2, 10.0


def _solve(name, fact, nu, strategy, batch, points, t, *, field="lotka_volterra", d=2, constraint="ts0", prior="iwp",
           rtol=1e-6, mu=1.0):
    return {"name": name, "kind": "solve", "fact": fact, "nu": nu, "strategy": strategy, "batch": batch,
            "points": points, "t": t, "field": field, "d": d, "constraint": constraint, "prior": prior, "rtol": rtol,
            "mu": mu}


def listed():
    return [
        # one solve of the quickstart problem through the mirrored API: what a user who
        # switches from the reference runs first, and what latency-bound callers run
        _solve("plain_dense_filter", "dense", 4, "filter", 1, 200, 50.0),
        # the same for a smoother of an isotropic model
        _solve("plain_isotropic_smoother", "isotropic", 4, "fixedpoint", 1, 200, 50.0),
        # the benchmark's headline batch: uneven lengths, smoothed on 200 points
        _solve("batch_isotropic_smoother", "isotropic", 4, "fixedpoint", 4096, 200, 50.0),
        # terminal-value style filtering of an odd, middling batch (simulation-based inference)
        _solve("batch_isotropic_filter", "isotropic", 3, "filter", 777, 5, 30.0),
        # the quickstart configuration over a batch: dense state, 200 points
        _solve("batch_dense_filter", "dense", 4, "filter", 1024, 200, 50.0),
        # stiff problems need the dense Jacobian: van der Pol, terminal values
        _solve("batch_dense_stiff", "dense", 5, "filter", 1024, 2, 6.3, field="van_der_pol", constraint="ts1",
               rtol=1e-5, mu=100.0),
        # a Matern prior: a transition by matrix exponential in every step
        _solve("batch_dense_matern", "dense", 4, "filter", 200, 20, 30.0, prior="matern"),
        # a discretised PDE: one block per grid point, terminal values
        _solve("batch_blockdiag_pde", "blockdiag", 2, "filter", 256, 2, 1.0, field="burgers", d=512, rtol=1e-4),
        # parameter estimation: log-likelihood and gradient of 101 observations on a 2001-point grid
        {"name": "lml_gradient_forward", "kind": "lml", "nu": 3, "batch": 1024, "steps": 2000, "every": 20,
         "gradient": "forward"},
        # the same by the adjoint, which does not grow with the number of parameters
        {"name": "lml_gradient_reverse", "kind": "lml", "nu": 3, "batch": 1024, "steps": 2000, "every": 20,
         "gradient": "reverse"},
        # dense output of finished smoothing solutions
        {"name": "offgrid_marginals", "kind": "offgrid", "nu": 4, "strategy": "fixedinterval", "batch": 4096,
         "points": 200, "queries": 256},
        # sample paths of finished smoothing solutions
        {"name": "posterior_samples", "kind": "sample", "nu": 4, "batch": 4096, "points": 200, "samples": 16},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["isotropic", "isotropic", "dense", "dense", "stiff", "matern", "blockdiag", "lml", "lml", "offgrid",
                       "sample"])
    t = round(rng.uniform(10.0, 50.0), 3)
    rtol = round(10.0 ** rng.uniform(-6.0, -4.0), 9)
    if kind == "isotropic":
        c = _solve("", "isotropic", rng.choice([3, 3, 4, 4, 4, 2, 5]), rng.choice(["filter", "fixedpoint", "fixedpoint"]),
                   _log_int(rng, 1, 4096), _log_int(rng, 2, 200), t, rtol=rtol)
    elif kind == "dense":
        c = _solve("", "dense", rng.choice([2, 3, 4, 4, 5]), rng.choice(["filter", "filter", "fixedpoint"]),
                   _log_int(rng, 1, 1024), _log_int(rng, 2, 200), t, rtol=rtol, constraint=rng.choice(["ts0", "ts1"]))
    elif kind == "stiff":
        c = _solve("", "dense", rng.choice([3, 4, 5]), "filter", _log_int(rng, 1, 1024), _log_int(rng, 2, 50), 6.3,
                   field="van_der_pol", constraint="ts1", rtol=max(rtol, 1e-5), mu=round(rng.uniform(5.0, 100.0), 2))
    elif kind == "matern":
        c = _solve("", "dense", rng.choice([2, 3, 4]), "filter", _log_int(rng, 1, 200), _log_int(rng, 2, 20),
                   min(t, 30.0), rtol=rtol, prior="matern")
    elif kind == "blockdiag":
        d = _log_int(rng, 5, 512)
        c = _solve("", "blockdiag", 2, "filter", _log_int(rng, 1, 256), _log_int(rng, 2, 10),
                   round(rng.uniform(0.05, 0.3), 3), field="burgers", d=d, rtol=max(rtol, 1e-5))
    elif kind == "lml":
        every = rng.choice([10, 20, 25])
        c = {"kind": "lml", "nu": rng.choice([3, 3, 4]), "batch": _log_int(rng, 1, 1024),
             "steps": every * _log_int(rng, 10, 2000 // every), "every": every,
             "gradient": rng.choice(["forward", "reverse"])}
    elif kind == "offgrid":
        c = {"kind": "offgrid", "nu": rng.choice([3, 4]), "strategy": rng.choice(["filter", "fixedinterval"]),
             "batch": _log_int(rng, 16, 4096), "points": _log_int(rng, 20, 200), "queries": _log_int(rng, 8, 256)}
    else:
        c = {"kind": "sample", "nu": rng.choice([3, 4]), "batch": _log_int(rng, 16, 4096),
             "points": _log_int(rng, 20, 200), "samples": _log_int(rng, 1, 16)}
    c.pop("name", None)
    return c


# ---------------------------------------------------------------- inputs
def _device():
    return torch.device("cuda")


def _dev(x):
    return torch.as_tensor(np.ascontiguousarray(x), dtype=F64, device=_device())


def _lv_inputs(batch, seed):
    rng = np.random.default_rng(seed)
    params = THETA0 * np.exp(rng.uniform(np.log(0.8), np.log(1.2), size=(batch, 4)))
    return rng, params, rng.uniform(10.0, 30.0, size=(batch, 2))


def _solve_inputs(case, seed):
    """(params, y0, save_at) of a solve case, numpy float64."""
    B, K, d = case["batch"], case["points"], case["d"]
    if case["field"] == "lotka_volterra":
        rng, params, y0 = _lv_inputs(B, seed)
        t_end = case["t"] * rng.uniform(0.4, 1.6, size=B) if B > 1 else np.full(1, case["t"])
    elif case["field"] == "van_der_pol":
        rng = np.random.default_rng(seed)
        params = np.exp(rng.uniform(0.0, np.log(case["mu"]), size=(B, 1)))
        y0 = np.tile([2.0, 0.0], (B, 1)) + rng.uniform(-0.1, 0.1, size=(B, 2)) * [1.0, 0.0]
        t_end = np.full(B, case["t"])
    else:
        rng = np.random.default_rng(seed)
        k = np.arange(1, 9)
        amp = rng.normal(size=(B, 8)) / k
        y0 = amp @ np.sin(2 * np.pi * k[:, None] * np.arange(d) / d)
        params = np.tile([0.01, 1.0 / d], (B, 1))
        t_end = np.full(B, case["t"])
    return params, y0, t_end[:, None] * np.linspace(0.0, 1.0, K)


def _matern_drift(N, d, length_scale=10.0):
    z = math.sqrt(2 * (N - 0.5)) / length_scale
    return np.concatenate([-math.comb(N, i) * z ** (N - i) * np.eye(d) for i in range(N)], axis=1)


def _solve_config(case):
    drift = None
    if case["prior"] == "matern":
        drift = _dev(_matern_drift(case["nu"] + 1, case["d"]))
    return capi.Config(
        factorisation=case["fact"], num_derivatives=case["nu"], ode_dim=case["d"], constraint=case["constraint"],
        strategy=case["strategy"], solver="dynamic", vector_field=case["field"],
        n_params={"lotka_volterra": 4, "van_der_pol": 1, "burgers": 2}[case["field"]], rtol=case["rtol"],
        atol=1e-2 * case["rtol"], dt0=DT0 if case["field"] != "burgers" else 1e-3,
        prior="iwp" if drift is None else "exponential", prior_drift=drift)


def _lml_inputs(case, seed):
    """(params, y0, grid, data, stds): noisy observations of each instance's solution (RK4 on the grid),
    the likelihood evaluated near the parameters a fit starts from."""
    rng, params, y0 = _lv_inputs(case["batch"], seed)
    n, every = case["steps"], case["every"]
    h = 0.01
    u = y0.T.copy()
    a, b, c, e = params.T

    def f(u):
        return np.stack([a * u[0] - b * u[0] * u[1], -c * u[1] + e * u[0] * u[1]])

    obs = [u.copy()]
    for i in range(1, n + 1):
        k1 = f(u)
        k2 = f(u + 0.5 * h * k1)
        k3 = f(u + 0.5 * h * k2)
        k4 = f(u + h * k3)
        u = u + h / 6.0 * (k1 + 2 * k2 + 2 * k3 + k4)
        if i % every == 0:
            obs.append(u.copy())
    data = np.stack(obs).transpose(2, 0, 1)
    stds = 0.1 * np.sqrt(np.mean(data**2, axis=-1))
    data = data + 0.1 * np.abs(data) * rng.normal(size=data.shape)
    start = THETA0 * np.exp(rng.uniform(-0.02, 0.02, size=params.shape))
    return start, rng.uniform(19.0, 21.0, size=y0.shape), h * np.arange(n + 1), data, stds[..., None]


def _posterior_inputs(case, seed):
    """(config, params, y0, times) of the solve whose solution an off-grid or sampling case works on."""
    rng, params, y0 = _lv_inputs(case["batch"], seed)
    strategy = case.get("strategy", "fixedinterval")
    cfg = capi.Config(factorisation="isotropic", num_derivatives=case["nu"], ode_dim=2, strategy=strategy, solver="dynamic")
    t_end = rng.uniform(20.0, 80.0, size=case["batch"]) * case["points"] / 200.0
    return rng, cfg, params, y0, t_end[:, None] * np.linspace(0.0, 1.0, case["points"])


def _prepare_solve(case, seed):
    params, y0, save_at = _solve_inputs(case, seed)
    cfg = _solve_config(case)
    P, Y0, T = _dev(params), _dev(y0), _dev(save_at)
    if case["batch"] > 1 or case["fact"] == "blockdiag" or case["field"] != "lotka_volterra" or case["prior"] != "iwp":
        tc = capi.taylor_coefficients(case["field"], P, Y0, 0.0, case["nu"])
        return {"kind": "solve", "cfg": cfg, "params": P, "tcoeffs": tc, "save_at": T}
    # one instance: the mirrored API, as the quickstart uses it
    vf = pdq.lotka_volterra(*[float(x) for x in params[0]])
    tcoeffs, _ = pdq.jetexpand_ode_padded_scan(num=case["nu"])(vf, [Y0[0]], t=0.0)
    ssm = pdq.state_space_model_dense() if case["fact"] == "dense" else pdq.state_space_model_isotropic()
    ts = ssm.constraint_ode_ts0(vf) if case["constraint"] == "ts0" else ssm.constraint_ode_ts1(vf)
    strategy = pdq.strategy_filter() if case["strategy"] == "filter" else pdq.strategy_smoother_fixedpoint()
    solver = pdq.solver_dynamic(strategy=strategy, constraint=ts)
    solve = ivpsolve.solve_adaptive_save_at(solver=solver, error=pdq.error_residual_std(constraint=ts))
    return {"kind": "plain", "solve": solve, "init": ssm.prior_wiener_integrated(tcoeffs), "save_at": T[0],
            "rtol": case["rtol"], "atol": 1e-2 * case["rtol"], "smoother": case["strategy"] != "filter"}


def prepare(case, seed):
    if case["kind"] == "solve":
        return _prepare_solve(case, seed)
    if case["kind"] == "lml":
        params, y0, grid, data, stds = _lml_inputs(case, seed)
        problem = torch_ops.LMLProblem("lotka_volterra", case["nu"], 2, _dev(grid), case["every"], lml_gradient=case["gradient"])
        return {"kind": "lml", "problem": problem, "params": _dev(params).requires_grad_(),
                "y0": _dev(y0).requires_grad_(), "data": _dev(data), "stds": _dev(stds)}
    rng, cfg, params, y0, times = _posterior_inputs(case, seed)
    P, T = _dev(params), _dev(times)
    tc = capi.taylor_coefficients("lotka_volterra", P, _dev(y0), 0.0, case["nu"])
    out = capi.solve(cfg, P, tc, T, fixed_grid=True)
    if case["kind"] == "offgrid":
        q = np.sort(rng.uniform(0.0, 1.0, size=(case["batch"], case["queries"])), axis=1) * times[:, -1:]
        return {"kind": "offgrid", "cfg": cfg, "solution": out, "times": T, "queries": _dev(q)}
    gen = torch.Generator(device=_device())
    gen.manual_seed(int(seed))
    base = torch.randn(case["batch"], case["samples"], case["points"], case["nu"] + 1, generator=gen, dtype=F64, device=_device())
    return {"kind": "sample", "cfg": cfg, "solution": out, "points": case["points"], "base": base}


# ------------------------------------------------------------------- run
def run(state):
    kind = state["kind"]
    if kind == "plain":
        sol = state["solve"](state["init"], save_at=state["save_at"], atol=state["atol"], rtol=state["rtol"])
        out = {"t": sol.t, "mean": sol.u.mean_flat, "chol": sol.u.cholesky_flat, "output_scale": sol.output_scale,
               "num_steps": sol.num_steps, "attempts": sol.attempts}
        if state["smoother"]:
            post = sol.solution_full.posterior
            out["cond_A"], out["cond_mean"] = post.conditional.A, post.conditional.noise.mean_flat
            out["cond_chol"] = post.conditional.noise.cholesky_flat
        return out
    if kind == "solve":
        return capi.solve(state["cfg"], state["params"], state["tcoeffs"], state["save_at"])
    if kind == "lml":
        value = torch_ops.lml(state["problem"], state["data"], state["stds"], params=state["params"], y0=state["y0"])
        g_params, g_y0 = torch.autograd.grad(value.sum(), (state["params"], state["y0"]))
        return {"value": value, "g_params": g_params, "g_y0": g_y0}
    if kind == "offgrid":
        mean, chol = capi.offgrid_marginals(state["cfg"], state["solution"], state["times"], state["queries"])
        return {"mean": mean, "chol": chol}
    return {"samples": capi.sample(state["cfg"], state["solution"], state["points"], state["base"])}


# ------------------------------------------------------------------ work
def _qr_flops(m, k):
    return 2.0 * m * k * k - 2.0 / 3.0 * k**3


def _attempts(case):
    """Typical step attempts of one instance (measured on such inputs; the order and the tolerance set them)."""
    if case["field"] == "burgers":
        return 25500.0 * (case["d"] / 512.0) ** 2 * case["t"] + 20.0
    if case["field"] == "van_der_pol":
        return 148.0 * (1e-5 / case["rtol"]) ** (1.0 / (case["nu"] + 1))
    return 12.5 * case["t"] * (1e-6 / case["rtol"]) ** (1.0 / (case["nu"] + 1)) * 1.6 ** (4 - case["nu"])


def work(case):
    if case["kind"] == "solve":
        N, d, B, K = case["nu"] + 1, case["d"], case["batch"], case["points"]
        nb, n, mc, ko = {"dense": (1, N * d, 1, d), "isotropic": (1, N, d, 1), "blockdiag": (d, N, 1, 1)}[case["fact"]]
        predict, update = 2.0 * n**3 + _qr_flops(2 * n, n), _qr_flops(n + ko, n + ko) + 2.0 * n * ko * (n + mc)
        if case["prior"] == "matern":
            predict += 12.0 * n**3 + 2.0 * n * n * (n + 10 * d) + _qr_flops(10 * d, n)
        revert = 2.0 * n**3 + _qr_flops(2 * n, 2 * n) + n**3
        merge = 4.0 * n**3 + _qr_flops(2 * n, n)
        smoother = case["strategy"] != "filter"
        attempt = (revert + merge if smoother else predict) + update + _qr_flops(n + ko, ko)
        point = 2.0 * (revert + merge) + predict if smoother else predict
        flops = B * nb * (_attempts(case) * attempt + (K - 1) * point)
        per_point = 2 + nb + nb * (n * mc + n * n)
        if smoother:  # filtering marginal and backward conditional, the latter read back once
            per_point += nb * (n * mc + n * n) + 2 * nb * (2 * n * n + n * mc + 2 * n)
        return {"bytes": 8.0 * B * (K * (1 + per_point) + (N + 2) * d), "flops": flops}
    N, B = case["nu"] + 1, case["batch"]
    revert = 2.0 * N**3 + _qr_flops(2 * N, 2 * N) + N**3
    merge = 4.0 * N**3 + _qr_flops(2 * N, N)
    if case["kind"] == "lml":
        nodes = case["steps"] // case["every"] + 1
        means = 12.0 * N * N * 2 * (7 if case["gradient"] == "forward" else 3)
        flops = B * (case["steps"] * (revert + merge + _qr_flops(N + 1, N + 1) + means) + nodes * (merge + means))
        return {"bytes": 8.0 * B * nodes * (2 * (2 * N * N + 4 * N) + 3), "flops": flops}
    if case["kind"] == "offgrid":
        q = B * case["queries"]
        smoother = case["strategy"] != "filter"
        flops = q * (2.0 * revert + merge if smoother else 2.0 * N**3 + _qr_flops(2 * N, N))
        read = B * case["points"] * (2 + (2 if smoother else 1) * (2 * N + N * N))
        return {"bytes": 8.0 * (read + q * (1 + 2 * N + N * N)), "flops": flops}
    s, K = B * case["samples"], case["points"]
    return {"bytes": 8.0 * (s * K * 3 * N + B * (K - 1) * (2 * N * N + 4 * N)), "flops": s * (K - 1) * (4.0 * N * N * 2)}


# ----------------------------------------------------------------- exact
def _iwp(N):
    """The preconditioned transition (binomials) and the Cholesky factor of its noise, 1 / (a_i + a_j + 1)
    with a_i = N - 1 - i, factored exactly in rationals up to the final square roots."""
    A = torch.zeros(N, N, dtype=F64)
    for i in range(N):
        for j in range(i, N):
            A[i, j] = math.comb(N - 1 - i, j - i)
    L = [[Fraction(0)] * N for _ in range(N)]
    D = [Fraction(0)] * N
    for j in range(N):
        for i in range(j, N):
            v = Fraction(1, 2 * (N - 1) - i - j + 1) - sum(L[i][k] * L[j][k] * D[k] for k in range(j))
            if i == j:
                D[j] = v
            L[i][j] = v / D[j]
    Q = torch.tensor([[float(L[i][j]) * math.sqrt(D[j]) for j in range(N)] for i in range(N)], dtype=F64)
    return A, Q


def _taylor(field, p, y0, num):
    """The solution's derivatives 0..num at the initial value (B, num + 1, d), by Cauchy products."""
    c = [y0]

    def product(a, b, i):
        return sum(a(c[j]) * b(c[i - j]) for j in range(i + 1))

    def x(u):
        return u[:, 0]

    def y(u):
        return u[:, 1]

    squares = []
    for i in range(num):
        if field == "lotka_volterra":
            xy = product(x, y, i)
            f = torch.stack([p[:, 0] * x(c[i]) - p[:, 1] * xy, -p[:, 2] * y(c[i]) + p[:, 3] * xy], dim=1)
        elif field == "van_der_pol":
            squares.append((1.0 if i == 0 else 0.0) - product(x, x, i))
            f = torch.stack([y(c[i]), p[:, 0] * sum(squares[j] * y(c[i - j]) for j in range(i + 1)) - x(c[i])], dim=1)
        else:
            dx = p[:, 1:2]
            um, up = c[i].roll(1, 1), c[i].roll(-1, 1)
            slope = product(lambda u: u, lambda u: u.roll(-1, 1) - u.roll(1, 1), i) / (2 * dx)
            f = -slope + p[:, :1] * (up - 2 * c[i] + um) / dx**2
        c.append(f / (i + 1))
    return torch.stack([c[i] * math.factorial(i) for i in range(num + 1)], dim=1)


def _r(A):
    """The upper-triangular factor (k x k) of the QR decomposition of a batch of m x k matrices."""
    A = A.clone()
    m, k = A.shape[-2:]
    for i in range(min(m - 1, k)):
        x = A[..., i:, i]
        a0 = x[..., 0]
        beta = -torch.copysign(torch.linalg.vector_norm(x, dim=-1), a0)
        den = torch.where(beta == 0, 1.0, a0 - beta)
        v = x / den[..., None]
        v[..., 0] = 1.0
        tau = torch.where(beta == 0, 0.0, (beta - a0) / torch.where(beta == 0, 1.0, beta))
        w = tau[..., None] * (v[..., None, :] @ A[..., i:, i:])[..., 0, :]
        A[..., i:, i:] -= v[..., :, None] * w[..., None, :]
    A = A.triu()
    if m < k:
        A = torch.cat([A, A.new_zeros(*A.shape[:-2], k - m, k)], dim=-2)
    return A[..., :k, :]


class _Model:
    """A state-space model of a batch: means (B, nb, n, mc), factors (B, nb, n, n)."""

    def __init__(self, fact, N, d, field, params, constraint="ts0", drift=None):
        self.fact, self.N, self.d, self.field, self.p, self.constraint = fact, N, d, field, params, constraint
        self.n, self.mc, self.ko = {"dense": (N * d, 1, d), "isotropic": (N, d, 1), "blockdiag": (N, 1, 1)}[fact]
        dev = params.device
        A, Q = _iwp(N)
        eye = torch.eye(d if fact == "dense" else 1, dtype=F64)
        self.A, self.Q = torch.kron(A, eye).to(dev), torch.kron(Q, eye).to(dev)
        self.pw = torch.arange(N - 1, -1, -1, dtype=F64).repeat_interleave(self.n // N).to(dev)
        self.fact_pw = torch.exp(torch.lgamma(self.pw + 1)).round()
        self.drift = None if drift is None else drift.to(dev)
        if drift is not None:
            x, w = np.polynomial.legendre.leggauss(14)
            self.nodes, self.weights = torch.tensor((x + 1) / 2, dtype=F64, device=dev), torch.tensor(w / 2, dtype=F64, device=dev)

    def state(self, tcoeffs):
        """(B, N, d) Taylor coefficients as a mean and a zero factor."""
        B = tcoeffs.shape[0]
        if self.fact == "isotropic":
            m = tcoeffs[:, None]
        elif self.fact == "dense":
            m = tcoeffs.reshape(B, 1, self.n, 1)
        else:
            m = tcoeffs.transpose(1, 2)[..., None]
        return m, torch.zeros(*m.shape[:2], self.n, self.n, dtype=F64, device=m.device)

    def coefficient(self, m, i):
        if self.fact == "isotropic":
            return m[:, 0, i]
        return m[:, 0, i * self.d : (i + 1) * self.d, 0] if self.fact == "dense" else m[:, :, i, 0]

    def flat(self, m):
        return m.reshape(m.shape[0], -1)

    def f(self, u):
        p = self.p
        if self.field == "lotka_volterra":
            xy = u[:, 0] * u[:, 1]
            return torch.stack([p[:, 0] * u[:, 0] - p[:, 1] * xy, -p[:, 2] * u[:, 1] + p[:, 3] * xy], dim=1)
        if self.field == "van_der_pol":
            return torch.stack([u[:, 1], p[:, 0] * (1.0 - u[:, 0] ** 2) * u[:, 1] - u[:, 0]], dim=1)
        um, up, dx = u.roll(1, 1), u.roll(-1, 1), p[:, 1:2]
        return -u * (up - um) / (2 * dx) + p[:, :1] * (up - 2 * u + um) / dx**2

    def jac(self, u):
        p = self.p
        if self.field == "lotka_volterra":
            rows = [[p[:, 0] - p[:, 1] * u[:, 1], -p[:, 1] * u[:, 0]], [p[:, 3] * u[:, 1], -p[:, 2] + p[:, 3] * u[:, 0]]]
        else:
            one = torch.ones_like(u[:, 0])
            rows = [[0 * one, one], [-2 * p[:, 0] * u[:, 0] * u[:, 1] - 1.0, p[:, 0] * (1 - u[:, 0] ** 2)]]
        return torch.stack([torch.stack(r, dim=1) for r in rows], dim=1)

    def linearise(self, m):
        """(H, b): the observation H x + b = 0 of the ODE at m."""
        B, nb = m.shape[:2]
        u = self.coefficient(m, 0)
        f = self.f(u)
        H = torch.zeros(B, nb, self.ko, self.n, dtype=F64, device=m.device)
        if self.fact == "dense":
            H[:, 0, :, self.d : 2 * self.d] = torch.eye(self.d, dtype=F64, device=m.device)
            b = -f[:, None, :, None]
            if self.constraint == "ts1":
                J = self.jac(u)
                H[:, 0, :, : self.d] = -J
                b = b + (J @ u[..., None])[:, None]
            return H, b
        H[..., 0, 1] = 1.0
        return H, -(f[:, None, None, :] if self.fact == "isotropic" else f[:, :, None, None])

    def transition(self, dt):
        """(P, A, W): preconditioner (B, 1, n), transition and unit-scale noise columns in preconditioned
        coordinates."""
        P = dt[:, None, None] ** self.pw / self.fact_pw
        root = dt.abs().sqrt()[:, None, None, None]
        if self.drift is None:
            return P, self.A, root * self.Q
        d, n = self.d, self.n
        F = torch.zeros(n, n, dtype=F64, device=dt.device)
        F[: n - d, d:] = torch.eye(n - d, dtype=F64, device=dt.device)
        F[n - d :] = self.drift
        Fp = dt[:, None, None] * F / P[:, 0, :, None] * P[:, 0, None, :]
        E = torch.linalg.matrix_exp(torch.cat([Fp[:, None], Fp[:, None] * self.nodes[:, None, None]], dim=1))
        noise = E[:, 1:, :, n - d :] / P[:, 0, None, None, n - d :] * self.weights.sqrt()[:, None, None]
        return P, E[:, :1], root * noise.permute(0, 2, 1, 3).reshape(len(dt), 1, n, -1)

    def predict(self, tr, s, m, L):
        P, A, W = tr
        PI = 1.0 / P[..., None]
        R = _r(torch.cat([(A @ (PI * L)).mT, (s * W).mT.expand(*L.shape[:2], -1, -1)], dim=-2))
        return P[..., None] * (A @ (PI * m)), P[..., None] * R.mT

    def revert(self, tr, s, m, L):
        """The prediction and the backward conditional x | x_next ~ N(G x_next + c, C C^T)."""
        P, A, W = tr
        n, PI = self.n, 1.0 / P[..., None]
        Lp, mp = PI * L, PI * m
        top = torch.cat([(s * W).mT.expand(*L.shape[:2], -1, -1), (A @ Lp).mT], dim=-2)
        right = torch.cat([torch.zeros_like(top[..., : W.shape[-1], :]), Lp.mT], dim=-2)
        R = _r(torch.cat([top, right], dim=-1))
        gain = torch.linalg.solve_triangular(R[..., :n, :n], R[..., :n, n:], upper=True).mT
        mo = A @ mp
        pred = (P[..., None] * mo, P[..., None] * R[..., :n, :n].mT)
        return pred, (P[..., None] * gain * PI.mT, P[..., None] * (mp - gain @ mo), P[..., None] * R[..., n:, n:].mT)

    def observe(self, H, b, m, L):
        R = _r((H @ L).mT)
        return H @ m + b, R.mT

    def update(self, H, noise, resid, m, L):
        """Condition on H x + resid - H m = 0 with observation noise factor `noise` (ko x ko)."""
        ko = self.ko
        top = torch.cat([noise.expand(*L.shape[:2], ko, ko), torch.zeros(*L.shape[:2], ko, self.n, dtype=F64, device=L.device)], dim=-1)
        R = _r(torch.cat([top, torch.cat([(H @ L).mT, L.mT], dim=-1)], dim=-2))
        gain = torch.linalg.solve_triangular(R[..., :ko, :ko], R[..., :ko, ko:], upper=True).mT
        return m - gain @ resid, R[..., ko:, ko:].mT, R[..., :ko, :ko].mT

    def whiten(self, om, oL):
        w = torch.linalg.solve_triangular(oL, om, upper=False)
        return torch.sqrt((w * w).sum(dim=(-2, -1)) / (self.ko * self.mc))

    @staticmethod
    def merge(first, second):
        G1, c1, L1 = first
        G2, c2, L2 = second
        return G1 @ G2, G1 @ c2 + c1, _r(torch.cat([(G1 @ L2).mT, L1.mT], dim=-2)).mT

    @staticmethod
    def through(cond, m, L):
        G, c, C = cond
        return G @ m + c, _r(torch.cat([(G @ L).mT, C.mT], dim=-2)).mT

    def identity(self, m):
        eye = torch.eye(self.n, dtype=F64, device=m.device).expand(*m.shape[:2], -1, -1)
        return eye.clone(), torch.zeros_like(m), torch.zeros_like(eye)


def _pick(mask, new, old):
    return [torch.where(mask.reshape(-1, *[1] * (x.dim() - 1)), x, y) for x, y in zip(new, old)]


def _exact_solve(case, seed):
    params, y0, save_at = (_dev(x) for x in _solve_inputs(case, seed))
    N, d, B, K = case["nu"] + 1, case["d"], case["batch"], case["points"]
    drift = torch.tensor(_matern_drift(N, d), dtype=F64) if case["prior"] == "matern" else None
    M = _Model(case["fact"], N, d, case["field"], params, case["constraint"], drift)
    smoother = case["strategy"] != "filter"
    rtol, atol = case["rtol"], 1e-2 * case["rtol"]
    m, L = M.state(_taylor(case["field"], params, y0, case["nu"]))
    t = save_at[:, 0].clone()
    dt = torch.full((B,), DT0 if case["field"] != "burgers" else 1e-3, dtype=F64, device=t.device)
    ident = M.identity(m)
    nb = m.shape[1]
    os = torch.ones(B, nb, dtype=F64, device=t.device)
    step = [t, m, L, os, *ident]  # step_from: t, mean, factor, output scale, conditional
    prev = list(step)  # interp_from
    k = torch.ones(B, dtype=torch.int64, device=t.device)
    means = torch.zeros(B, K, *m.shape[1:], dtype=F64, device=t.device)
    scales = torch.zeros(B, K, nb, dtype=F64, device=t.device)
    times = torch.zeros(B, K, dtype=F64, device=t.device)
    means[:, 0], scales[:, 0], times[:, 0] = m, os, t
    rows = torch.arange(B, device=t.device)

    def save(mask, t1, mean, scale):
        r, c = rows[mask], k[mask]
        means[r, c], scales[r, c], times[r, c] = mean[mask], scale[mask], t1[mask]

    for _ in range(200000):
        live = k < K
        if not bool(live.any()):
            break
        t1 = save_at.gather(1, k.clamp(max=K - 1)[:, None])[:, 0]
        attempt = live & (step[0] + EPS < t1)
        # one attempt of every instance that still has to reach its next point
        h = torch.where(attempt, dt, 1e-3)
        tr = M.transition(h)
        P, A, W = tr
        um, uL = P[..., None] * (A @ (step[1] / P[..., None])), P[..., None] * W
        H, b = M.linearise(um)
        om, oL = M.observe(H, b, um, uL.expand(B, nb, -1, -1))
        sigma = M.whiten(om, oL)
        s = sigma[..., None, None]
        if smoother:
            (pm, pL), cond = M.revert(tr, s, step[1], step[2])
            cond = M.merge(step[4:], cond)
        else:
            (pm, pL), cond = M.predict(tr, s, step[1], step[2]), step[4:]
        nm, nL, _ = M.update(H, torch.zeros(M.ko, M.ko, dtype=F64, device=t.device), H @ pm + b, pm, pL)
        std = sigma[..., None] * torch.linalg.vector_norm(oL, dim=-1)  # (B, nb, ko)
        u0, u1 = M.coefficient(step[1], 0), M.coefficient(nm, 0)
        ratio = std.reshape(B, -1) * h[:, None] / (atol + rtol * torch.maximum(u0.abs(), u1.abs()))
        power = torch.sqrt((ratio * ratio).mean(dim=1)) ** (-1.0 / N)
        dt = torch.where(attempt, torch.clamp(SAFETY * power, FACTOR_MIN, FACTOR_MAX) * h, dt)
        ok = attempt & (power >= 1.0)
        new = [step[0] + h, nm, nL, sigma, *cond]
        prev, step = _pick(ok, step, prev), _pick(ok, new, step)
        # points that an instance has stepped on or over
        done = live & ~(step[0] + EPS < t1)
        over = done & (step[0] > t1 + EPS)
        if bool(over.any()):
            s = step[3][..., None, None]
            h0, h1 = torch.where(over, t1 - prev[0], 1e-3), torch.where(over, step[0] - t1, 1e-3)
            if smoother:
                (im, iL), _ = M.revert(M.transition(h0), s, prev[1], prev[2])
                _, c1 = M.revert(M.transition(h1), s, im, iL)
            else:
                (im, iL), c1 = M.predict(M.transition(h0), s, prev[1], prev[2]), step[4:]
            save(over, t1, im, step[3])
            prev = _pick(over, [t1, im, iL, step[3], *ident], prev)
            step = _pick(over, [*step[:4], *c1], step)
        hit = done & ~over
        if bool(hit.any()):
            save(hit, step[0], step[1], step[3])
            prev = _pick(hit, [*step[:4], *(ident if smoother else step[4:])], prev)
            step = _pick(hit, [*step[:4], *(ident if smoother else step[4:])], step)
        k = k + done.to(k.dtype)
    shape = (B, K, -1)
    out = {"t": times, "output_scale": scales, "mean": means.reshape(shape)}
    if smoother:
        out["filt_mean"], out["mean"] = out["mean"], None
        out["term_mean"] = M.through(step[4:], step[1], step[2])[0].reshape(B, -1)
    return out


def _exact_plain(out, case):
    N, d, K = case["nu"] + 1, case["d"], case["points"]
    mean = out["mean"]
    if mean is not None:
        mean = mean[0].reshape(K, N * d) if case["fact"] == "dense" else mean[0].reshape(K, N, d)
    return {"t": out["t"][0], "output_scale": out["output_scale"][0, :, 0], "mean": mean}


def _exact_lml(case, seed):
    params, y0, grid, data, stds = (_dev(x) for x in _lml_inputs(case, seed))
    params.requires_grad_()
    y0.requires_grad_()
    N, B, every = case["nu"] + 1, case["batch"], case["every"]
    M = _Model("isotropic", N, 2, "lotka_volterra", params)
    m, L = M.state(_taylor("lotka_volterra", params, y0, case["nu"]))
    # the factors do not depend on the parameters (ts0, no calibration): one recursion for the batch
    L, fixed = L[:1], torch.zeros(1, 1, dtype=F64, device=L.device)
    cond, nodes = None, []
    zero = torch.zeros(1, 1, N, 2, dtype=F64, device=L.device)
    H0 = torch.zeros(1, 1, 1, N, dtype=F64, device=L.device)
    H0[..., 0, 1] = 1.0
    one = torch.ones(1, dtype=F64, device=L.device)
    for i in range(1, case["steps"] + 1):
        h = float(grid[i] - grid[i - 1])
        tr = M.transition(h * one)
        (_, pL), (G, _, C) = M.revert(tr, 1.0, zero, L)
        P, A, _ = tr
        pm = P[..., None] * (A @ (m / P[..., None]))
        back = (G, m - G @ pm, C)
        cond = back if cond is None else M.merge(cond, back)
        _, b = M.linearise(pm)
        _, L2, _ = M.update(H0, fixed, zero[..., :1, :], zero, pL)
        R = _r(torch.cat([(H0 @ pL).mT, pL.mT], dim=-1))
        gain = (R[..., :1, 1:] / R[..., :1, :1]).mT
        m, L = pm - gain @ (H0 @ pm + b), L2
        if i % every == 0:
            nodes.append(cond)
            cond = None
    value, H1 = 0.0, torch.zeros(1, 1, 1, N, dtype=F64, device=L.device)
    H1[..., 0, 0] = 1.0
    L = L.expand(B, 1, N, N)
    count = len(nodes) + 1
    for j in range(len(nodes), -1, -1):
        if j < len(nodes):
            G, cc, C = nodes[j]
            m, L = G @ m + cc, _r(torch.cat([(G @ L).mT, C.mT.expand(B, 1, N, N)], dim=-2)).mT
        resid = m[:, :, :1] - data[:, j, None, None, :]
        m, L, oL = M.update(H1.expand(B, 1, 1, N), stds[:, j, :, None, None], resid, m, L)
        oL = oL[:, 0, 0, 0]
        white = (resid[:, 0, 0] / oL[:, None]).square().sum(dim=1)
        value = value - 0.5 * (white + 2 * (2.0 * torch.log(oL.abs()) + math.log(2 * math.pi)))
    value = value / count
    g_params, g_y0 = torch.autograd.grad(value.sum(), (params, y0))
    return {"value": value.detach(), "g_params": g_params, "g_y0": g_y0}


def _exact_offgrid(case, seed):
    s = prepare(case, seed)
    out, times, tq = s["solution"], s["times"], s["queries"]
    N, B, Q = case["nu"] + 1, case["batch"], case["queries"]
    i = torch.searchsorted(times, tq).clamp(1, case["points"] - 1)
    result = torch.empty(B, Q, 2 * N, dtype=F64, device=times.device)
    smoother = case["strategy"] != "filter"
    kind = "filt_" if smoother else ""
    for q in range(Q):  # one query of every instance at a time
        r, c = torch.arange(B, device=times.device), i[:, q]
        M = _Model("isotropic", N, 2, "lotka_volterra", torch.zeros(B, 4, dtype=F64, device=times.device))
        m = out[kind + "mean"][r, c - 1].reshape(B, 1, N, 2)
        L = out[kind + "chol"][r, c - 1].reshape(B, 1, N, N)
        sc = out["output_scale"].reshape(B, -1)[r, c][:, None, None, None]
        tr = M.transition(tq[:, q] - times[r, c - 1])
        if not smoother:
            result[:, q] = M.predict(tr, sc, m, L)[0].reshape(B, -1)
            continue
        (m, L), _ = M.revert(tr, sc, m, L)
        _, (G, cc, _) = M.revert(M.transition(times[r, c] - tq[:, q]), sc, m, L)
        result[:, q] = (G @ out["mean"][r, c].reshape(B, 1, N, 2) + cc).reshape(B, -1)
    return {"mean": result}


def _exact_sample(case, seed):
    s = prepare(case, seed)
    out, base = s["solution"], s["base"]
    N, B, K, S = case["nu"] + 1, case["batch"], case["points"], case["samples"]
    x = out["term_mean"].reshape(B, 1, N, 2) + (out["term_chol"].reshape(B, 1, N, N) @ base[:, :, K - 1, :, None])
    path = [x]
    for j in range(K - 2, -1, -1):
        A, C = out["cond_A"][:, j].reshape(B, 1, N, N), out["cond_chol"][:, j].reshape(B, 1, N, N)
        tl, to = out["cond_tl"][:, j].reshape(B, 1, N, 1), out["cond_to"][:, j].reshape(B, 1, N, 1)
        mean = to * (A @ (tl * x)) + out["cond_mean"][:, j].reshape(B, 1, N, 2)
        x = mean + to.abs() * (C @ base[:, :, j, :, None])
        path.append(x)
    return {"samples": torch.stack(path[::-1], dim=2).reshape(B, S, K, 2 * N)}


def exact(case, seed):
    if case["kind"] == "solve":
        # tens of thousands of attempts of a large PDE would take minutes
        if case["fact"] == "blockdiag" and _attempts(case) > 1500:
            return None
        out = _exact_solve(case, seed)
        mirrored = case["batch"] == 1 and case["fact"] != "blockdiag" and case["field"] == "lotka_volterra" and case["prior"] == "iwp"
        return _exact_plain(out, case) if mirrored else out
    return {"lml": _exact_lml, "offgrid": _exact_offgrid, "sample": _exact_sample}[case["kind"]](case, seed)
