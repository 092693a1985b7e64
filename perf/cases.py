"""Timed cases of geomjax_amd: one call each through a public entry point.

A case is a dict of plain values; ``prepare`` makes what a sampling program has
in hand (the model on the GPU, the chains' state, the transition's normals and
uniforms), ``run`` is one call, ``exact`` the same numbers in 64-bit torch.

Kinds:
  funnel_rmhmc   RMHMC with the Monge metric on Neal's funnel
  funnel_lmc     Lagrangian Monte Carlo with the Monge metric on the funnel
  rmhmc          RMHMC with the Fisher metric on one logistic posterior
  batch          the same on many posteriors of uneven sizes in one launch
  lmc            Lagrangian Monte Carlo with the Fisher metric
  mmala          manifold MALA with the Fisher metric
  nuts           NUTS over the RMHMC integrator, Fisher metric
  tangent        objective and derivative for tuning the step size by gradient
  ess            effective sample size and R-hat of a sample array

The accept uniforms lie in (0, 0.5): chains of these step sizes accept with a
higher probability than that nearly always, so that no decision hangs on the
last digit of an energy.
"""
import functools
import math
import random

import torch

import geomjax_amd as gj
from geomjax_amd.adjoint import esjd_acceptance
from geomjax_amd.nuts import NUTSNoise
from geomjax_amd.rmhmc import implicit_midpoint

DEV = "cuda:0"
F64 = torch.float64
PRIOR_VAR = 100.0
LOG2PI = math.log(2.0 * math.pi)


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------


def listed():
    return [
        # the smallest: four chains, one transition per call, as the funnel example runs
        {"name": "funnel_rmhmc_4x10_f64", "kind": "funnel_rmhmc", "dtype": "float64", "C": 4, "D": 10, "T": 1,
         "L": 16, "iters": 8, "eps": 0.05},
        # thousands of funnel chains, several transitions per persistent launch
        {"name": "funnel_rmhmc_8192x100_f32", "kind": "funnel_rmhmc", "dtype": "float32", "C": 8192, "D": 100,
         "T": 2, "L": 32, "iters": 8, "eps": 0.03},
        {"name": "funnel_lmc_8192x100_f32", "kind": "funnel_lmc", "dtype": "float32", "C": 8192, "D": 100, "T": 4,
         "L": 32, "eps": 0.03},
        # an ordinary small regression with odd sizes, one transition per call
        {"name": "rmhmc_777x23_c300_f32", "kind": "rmhmc", "dtype": "float32", "N": 777, "D": 23, "C": 300, "T": 1,
         "L": 10, "iters": 6, "eps": 0.1},
        # the headline workload: 2048 x 64, thousands of chains, float32 state
        {"name": "rmhmc_2048x64_c4096_f32", "kind": "rmhmc", "dtype": "float32", "N": 2048, "D": 64, "C": 4096,
         "T": 2, "L": 10, "iters": 6, "eps": 0.1},
        # the same posterior in float64
        {"name": "rmhmc_2048x64_c1024_f64", "kind": "rmhmc", "dtype": "float64", "N": 2048, "D": 64, "C": 1024,
         "T": 1, "L": 10, "iters": 6, "eps": 0.1},
        # many posteriors of 8..128 features and 256..4096 rows, 32 chains each
        {"name": "batch_64x32_f32", "kind": "batch", "dtype": "float32", "P": 64, "shapes": 3, "per": 32, "T": 1,
         "L": 10, "iters": 6, "eps": 0.1},
        # the explicit integrator with the Fisher metric
        {"name": "lmc_2048x64_c1024_f32", "kind": "lmc", "dtype": "float32", "N": 2048, "D": 64, "C": 1024, "T": 1,
         "L": 10, "eps": 0.1},
        # tree building: one NUTS transition of each chain
        {"name": "nuts_2048x64_c256_f64", "kind": "nuts", "dtype": "float64", "N": 2048, "D": 64, "C": 256, "M": 4,
         "iters": 6, "eps": 0.1},
        # manifold MALA, several transitions per launch
        {"name": "mmala_2048x64_c1024_f64", "kind": "mmala", "dtype": "float64", "N": 2048, "D": 64, "C": 1024,
         "T": 4, "eps": 0.3},
        # the derivative that tunes the step size
        {"name": "tangent_2048x64_c1024_f32", "kind": "tangent", "dtype": "float32", "N": 2048, "D": 64, "C": 1024,
         "L": 16, "iters": 6, "eps": 0.1},
        # convergence diagnostics over a window of samples of all chains
        {"name": "ess_100x4096x64_f32", "kind": "ess", "dtype": "float32", "T": 100, "C": 4096, "D": 64},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        c = _draw(rng)
        if _cost(c) <= _LARGEST[c["dtype"]]:
            return c


# flops of the costliest listed logistic case of each data type (float64 costs about ten times float32)
_LARGEST = {"float32": 2.0e13, "float64": 2.4e12}


def _cost(c):
    """Flops of a drawn case with narrow posteriors counted as 64 features and
    wide ones twice as 128."""
    if "N" not in c:
        return 0.0
    return work(dict(c, D=64))["flops"] if c["D"] <= 64 else 2.0 * work(dict(c, D=128))["flops"]


def _draw(rng):
    kind = rng.choice(["funnel_rmhmc", "funnel_lmc", "rmhmc", "rmhmc", "batch", "lmc", "nuts", "mmala", "tangent",
                       "ess"])
    f32 = rng.random() < 0.6
    c = {"kind": kind, "dtype": "float32" if f32 else "float64"}
    if kind in ("funnel_rmhmc", "funnel_lmc"):
        c.update(C=_log_int(rng, 1, 8192), D=_log_int(rng, 3, 128), T=_log_int(rng, 1, 4), L=rng.randint(4, 32),
                 eps=rng.choice([0.02, 0.03, 0.05]))
        if kind == "funnel_rmhmc":
            c["iters"] = rng.randint(4, 8)
        return c
    if kind == "ess":
        c.update(T=_log_int(rng, 20, 200), C=_log_int(rng, 2, 4096), D=_log_int(rng, 1, 128))
        return c
    if kind == "batch":
        c.update(dtype="float32", P=rng.randint(2, 64), shapes=rng.randint(0, 9999), per=rng.randint(1, 32), T=1,
                 L=rng.randint(4, 10), iters=6, eps=0.1)
        return c
    wide = 128 if kind == "rmhmc" else 64
    c.update(D=_log_int(rng, 2, wide), C=_log_int(rng, 1, 2048))
    c["N"] = max(4 * c["D"], _log_int(rng, 100, 4096))
    if kind == "rmhmc":
        c.update(T=rng.randint(1, 2), L=rng.randint(4, 10), iters=rng.randint(4, 8), eps=0.1)
    elif kind == "lmc":
        c.update(T=1, L=rng.randint(4, 10), eps=0.1)
    elif kind == "mmala":
        c.update(dtype="float64", T=rng.randint(1, 4), eps=0.3)
    elif kind == "nuts":
        c.update(dtype="float64", C=min(c["C"], 512), M=rng.randint(2, 4), iters=6, eps=0.1)
    else:
        c.update(dtype="float32", L=rng.randint(4, 16), iters=6, eps=0.1)
    return c


def tolerance(case):
    """Relative 2-norm errors per output, about four times what the present form
    differs from ``exact`` by over these ranges; the largest single difference
    (``max``) belongs to a chain in the funnel's neck or to the acceptance of a
    chain with a large energy error."""
    kind = case["kind"]
    if kind == "ess":
        return {"rel": 1e-6}
    if case["dtype"] == "float64":
        return {"rel": 2e-8, "max": 1e-5, "differ": 0.002}
    if kind == "funnel_rmhmc":  # the neck of the funnel amplifies a rounding most
        return {"rel": 2e-2, "max": 0.99, "differ": 0.002}
    if kind == "funnel_lmc":  # 1e-3 in the acceptance
        return {"rel": 4e-3, "max": 0.5, "differ": 0.002}
    if kind == "lmc":  # 3e-3 in the acceptance (four float32 log-determinants a step)
        return {"rel": 1.2e-2, "max": 0.5, "differ": 0.002}
    if kind == "tangent":
        return {"rel": 5e-3, "max": 0.5, "differ": 0.002}
    return {"rel": 1e-4, "differ": 0.002}


def _shapes(case):
    """(N, D) of every posterior of a batch."""
    r = random.Random(case["shapes"])
    return [(_log_int(r, 256, 4096), r.choice([8, 16, 32, 64, 128])) for _ in range(case["P"])]


def work(case):
    """Bytes: the state read and written, the normals, the samples and the data
    set once.  Flops: the contractions of the algorithm's metric evaluations (the
    Gram X^T diag X and the quadratic forms x^T G^-1 x, 2 N D^2 each), or for the
    funnel the per-coordinate arithmetic of an evaluation."""
    kind = case["kind"]
    b = 4 if case["dtype"] == "float32" else 8
    if kind == "batch":
        f = byts = 0.0
        for N, D in _shapes(case):
            one = work(dict(case, kind="rmhmc", N=N, D=D, C=case["per"]))
            f += one["flops"]
            byts += one["bytes"]
        return {"bytes": byts, "flops": f}
    C, D, T = case["C"], case["D"], case.get("T", 1)
    if kind == "ess":
        return {"bytes": float(T) * C * D * b, "flops": float(C) * D * 10 * T * math.log2(2 * T)}
    moved = b * C * D * (4 + 2 * T)
    if kind == "funnel_rmhmc":
        return {"bytes": float(moved), "flops": float(C) * T * case["L"] * (case["iters"] + 2) * (33 * D + 26)}
    if kind == "funnel_lmc":
        return {"bytes": float(moved), "flops": float(C) * T * case["L"] * 75 * D}
    N = case["N"]
    moved += b * N * (D + 1)
    gram = 2.0 * N * D * D
    if kind == "rmhmc":
        f = C * T * case["L"] * (case["iters"] + 1) * 2 * gram
    elif kind == "lmc":
        f = C * T * case["L"] * 6 * gram
    elif kind == "mmala":
        f = C * T * 5 * gram
    elif kind == "nuts":
        f = C * (2 ** case["M"] - 1) * (case["iters"] + 1) * 2 * gram
    else:
        f = C * case["L"] * (case["iters"] + 1) * 4 * gram
    return {"bytes": float(moved), "flops": float(f)}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------


def _dtype(case):
    return torch.float32 if case["dtype"] == "float32" else F64


def _posterior(g, N, D, chains):
    """X [N, D] iid N(0, 1/D), y from a true coefficient vector, and positions of
    ``chains`` chains spread as the posterior is (its normal approximation)."""
    X = torch.randn(N, D, generator=g, device=DEV, dtype=F64) / math.sqrt(D)
    beta = torch.randn(D, generator=g, device=DEV, dtype=F64)
    y = (torch.rand(N, generator=g, device=DEV, dtype=F64) < torch.sigmoid(X @ beta)).to(F64)
    z = torch.randn(chains, D, generator=g, device=DEV, dtype=F64)
    for _ in range(6):
        s = torch.sigmoid(X @ beta)
        chol = torch.linalg.cholesky((X.T * (s * (1 - s))) @ X + torch.eye(D, device=DEV, dtype=F64) / PRIOR_VAR)
        grad = X.T @ (y - s) - beta / PRIOR_VAR
        beta = beta + torch.cholesky_solve(grad[:, None], chol)[:, 0]
    q = beta + torch.linalg.solve_triangular(chol.T, z.T.contiguous(), upper=True).T
    return X, y, q.contiguous()


def _inputs(case, seed):
    """Plain tensors of a case: data sets, positions, normals and uniforms."""
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 1000003 + 17)
    dt = _dtype(case)
    kind = case["kind"]
    if kind == "ess":
        T, C, D = case["T"], case["C"], case["D"]
        x = torch.empty(T, C, D, device=DEV, dtype=dt)
        cur = torch.randn(C, D, generator=g, device=DEV, dtype=dt)
        for t in range(T):  # the autocorrelation of a well-tuned chain
            cur = 0.6 * cur + 0.8 * torch.randn(C, D, generator=g, device=DEV, dtype=dt)
            x[t] = cur
        return {"x": x}
    data = None
    if kind in ("funnel_rmhmc", "funnel_lmc"):
        C, D = case["C"], case["D"]
        q = torch.randn(C, D, generator=g, device=DEV, dtype=F64)
    elif kind == "batch":
        shapes = _shapes(case)
        C, D = case["P"] * case["per"], max(d for _, d in shapes)
        data = [_posterior(g, n, d, case["per"]) for n, d in shapes]
        q = torch.zeros(C, D, device=DEV, dtype=F64)
        for p, (_, _, qp) in enumerate(data):
            q[p * case["per"]:(p + 1) * case["per"], :qp.shape[1]] = qp
    else:
        C, D = case["C"], case["D"]
        data = [_posterior(g, case["N"], D, C)]
        q = data[0][2]
    T = case.get("T", 1)
    out = {"data": data, "q": q.to(dt)}
    out["z"] = torch.randn(T, C, D, generator=g, device=DEV, dtype=dt)
    out["u"] = 0.5 * torch.rand(T, C, generator=g, device=DEV, dtype=F64)
    if kind == "nuts":
        M = case["M"]
        out["tree"] = [torch.rand(C, n, generator=g, device=DEV, dtype=F64) for n in (M, M, 2 ** M - 1)]
    return out


def prepare(case, seed):
    inp = _inputs(case, seed)
    kind = case["kind"]
    if kind == "ess":
        return {"kind": kind, "x": inp["x"]}
    T, eps, L = case.get("T", 1), case["eps"], case.get("L", 0)
    fisher = gj.FisherMetric()
    key = gj.random.HostNoise(inp["z"], inp["u"]) if T > 1 else gj.random.HostNoise(inp["z"][0], inp["u"][0])
    st = {"kind": kind, "key": key, "T": T}
    if kind in ("funnel_rmhmc", "funnel_lmc"):
        model = gj.NealFunnel(case["D"])
    elif kind == "batch":
        model = gj.LogisticBatch([gj.LogisticRegression(X, y, PRIOR_VAR) for X, y, _ in inp["data"]], case["per"])
    else:
        model = gj.LogisticRegression(inp["data"][0][0], inp["data"][0][1], PRIOR_VAR)
    integrator = functools.partial(implicit_midpoint, max_iters=case["iters"]) if "iters" in case else None
    if kind == "funnel_rmhmc":
        alg = gj.rmhmc(model, eps, gj.MongeMetric(1.0), L, integrator=integrator)
    elif kind == "funnel_lmc":
        alg = gj.lmcmonge(model, eps, torch.ones(case["D"], device=DEV, dtype=_dtype(case)), L, alpha2=1.0)
    elif kind in ("rmhmc", "batch"):
        alg = gj.rmhmc(model, eps, fisher, L, integrator=integrator)
    elif kind == "lmc":
        alg = gj.lmc(model, eps, fisher, L)
    elif kind == "mmala":
        alg = gj.mmala(model, eps, fisher, reference_faithful=False)
    elif kind == "nuts":
        alg = gj.nuts(model, eps, fisher, max_num_doublings=case["M"], integrator=integrator)
        st["key"] = NUTSNoise(inp["z"][0], *inp["tree"])
    else:
        alg = gj.rmhmc(model, eps, fisher, L, integrator=integrator)
        st["tangent"] = functools.partial(_tangent, model=model, eps=eps, L=L, integrator=integrator)
    st["alg"] = alg
    st["state"] = alg.init(inp["q"])
    return st


def _tangent(key, state, model, eps, L, integrator):
    r = esjd_acceptance(key, state, model, eps, gj.FisherMetric(), L, integrator=integrator)
    return {"objective": r.objective, "acceptance": r.acceptance, "sq_jump": r.sq_jump,
            "d_objective": r.d_objective, "d_sq_jump": r.d_sq_jump}


def run(state):
    kind = state["kind"]
    if kind == "ess":
        x = state["x"]
        return {"ess": gj.ess(x, chain_axis=1, sample_axis=0), "rhat": gj.rhat(x, chain_axis=1, sample_axis=0)}
    if kind == "tangent":
        return state["tangent"](state["key"], state["state"])
    if kind == "nuts":
        new, info = state["alg"].step(state["key"], state["state"])
        return {"state": tuple(new), "momentum": info.momentum, "energy": info.energy,
                "left": info.trajectory_leftmost_state, "right": info.trajectory_rightmost_state,
                "acceptance": info.acceptance_rate, "steps": info.num_integration_steps}
    if state["T"] > 1:
        r = gj.sampling.run_chains(state["alg"], state["state"], state["T"], state["key"])
        return {"state": tuple(r.state), "samples": r.samples, "acceptance": r.acceptance_rate}
    new, info = state["alg"].step(state["key"], state["state"])
    p = info.proposal
    if kind == "mmala":
        return {"state": tuple(new), "proposal": tuple(p), "acceptance": info.acceptance_rate,
                "accepted": info.is_accepted}
    p = p.state
    return {"state": tuple(new), "draw": info[0], "energy": info.energy, "acceptance": info.acceptance_rate,
            "accepted": info.is_accepted, "end": (p.position, p.momentum, p.velocity, p.logdensity)}


# ---------------------------------------------------------------------------
# the same numbers in 64-bit torch
# ---------------------------------------------------------------------------


class _Logistic:
    """Bernoulli-logit likelihood, normal prior, Fisher metric; q [C, D]."""

    def __init__(self, X, y):
        self.X, self.Xt, self.y = X, X.T.contiguous(), y
        self.N, self.D = X.shape

    def logp_grad(self, q):
        eta = q @ self.Xt
        soft = torch.clamp(eta, min=0.0) + torch.log1p(torch.exp(-eta.abs()))
        logp = (self.y * eta - soft).sum(1) - 0.5 * (q * q).sum(1) / PRIOR_VAR - 0.5 * self.D * (
            LOG2PI + math.log(PRIOR_VAR))
        return logp, (self.y - torch.sigmoid(eta)) @ self.X - q / PRIOR_VAR

    def gram(self, d):
        """X^T diag(d_c) X of every chain."""
        return (self.Xt * d[:, None, :]) @ self.X

    def eye(self):
        return torch.eye(self.D, device=self.X.device, dtype=F64)

    def geometry(self, q):
        """s, lambda, G, chol(G), G^-1 and a_n = x_n^T G^-1 x_n."""
        s = torch.sigmoid(q @ self.Xt)
        lam = s * (1 - s)
        G = self.gram(lam) + self.eye() / PRIOR_VAR
        chol = torch.linalg.cholesky(G)
        inv_chol = torch.linalg.solve_triangular(chol, self.eye().expand_as(G), upper=False)
        Gi = inv_chol.transpose(1, 2).contiguous() @ inv_chol
        a = ((Gi @ self.Xt) * self.Xt).sum(1)
        return s, lam, G, chol, Gi, a

    def draw(self, q, z):
        return (self.geometry(q)[3] @ z[..., None])[..., 0]

    def field(self, q, p):
        s, lam, _, _, Gi, a = self.geometry(q)
        u = (Gi @ p[..., None])[..., 0]
        b = u @ self.Xt
        h = 0.5 * lam * (1 - 2 * s) * (a - b * b) - (self.y - s)
        return u, h @ self.X + q / PRIOR_VAR

    def energy(self, q, p):
        _, _, _, chol, Gi, _ = self.geometry(q)
        u = (Gi @ p[..., None])[..., 0]
        logdet = 2 * torch.log(torch.diagonal(chol, dim1=1, dim2=2)).sum(1)
        return -self.logp_grad(q)[0] + 0.5 * (p * u).sum(1) + 0.5 * logdet + 0.5 * self.D * LOG2PI, u


class _Funnel:
    """Neal's funnel (log scale last, sigma = 3) with G = I + g g^T."""

    sigma2 = 9.0

    def __init__(self, D):
        self.D = D

    def logp_grad(self, q):
        x, v = q[:, :-1], q[:, -1]
        n = self.D - 1
        e, sx = torch.exp(-v), (x * x).sum(1)
        logp = -0.5 * v * v / self.sigma2 - math.log(3.0) - 0.5 * LOG2PI - 0.5 * e * sx - 0.5 * n * (v + LOG2PI)
        gv = -v / self.sigma2 - 0.5 * n + 0.5 * e * sx
        return logp, torch.cat([-e[:, None] * x, gv[:, None]], 1)

    def hvp(self, q, w):
        x, v = q[:, :-1], q[:, -1]
        e, sx = torch.exp(-v), (x * x).sum(1)
        hx = e[:, None] * (x * w[:, -1:] - w[:, :-1])
        hv = e * (x * w[:, :-1]).sum(1) - (1 / self.sigma2 + 0.5 * e * sx) * w[:, -1]
        return torch.cat([hx, hv[:, None]], 1)

    def draw(self, q, z):
        g = self.logp_grad(q)[1]
        G = torch.eye(self.D, device=q.device, dtype=F64) + g[:, :, None] * g[:, None, :]
        return (torch.linalg.cholesky(G) @ z[..., None])[..., 0]

    def field(self, q, p):
        g = self.logp_grad(q)[1]
        L = 1 + (g * g).sum(1)
        gp = (g * p).sum(1)
        u = p - (gp / L)[:, None] * g
        return u, self.hvp(q, g - gp[:, None] * u) / L[:, None] - g

    def energy(self, q, p):
        logp, g = self.logp_grad(q)
        gg, gp = (g * g).sum(1), (g * p).sum(1)
        perp = p - (gp / gg)[:, None] * g
        quad = (p * p).sum(1) / (1 + gg) + gg / (1 + gg) * (perp * perp).sum(1)
        u = p - (gp / (1 + gg))[:, None] * g
        return -logp + 0.5 * quad + 0.5 * torch.log1p(gg) + 0.5 * self.D * LOG2PI, u


def _midpoint(m, q, p, eps, iters):
    """One implicit-midpoint step: fixed-point iteration per chain, then the
    explicit half step from the last iterate."""
    h = 0.5 * eps

    def image(x):
        u, dH = m.field(*x)
        new = (q + h * u, p - h * dH)
        return new, torch.maximum((new[0] - x[0]).abs().amax(1), (new[1] - x[1]).abs().amax(1))

    x, norm = image((q, p))
    for _ in range(iters):
        active = torch.isfinite(norm) & (norm < 1e10) & (norm > 1e-6)
        if not bool(active.any()):
            break
        new, n1 = image(x)
        x = tuple(torch.where(active[:, None], a, b) for a, b in zip(new, x))
        norm = torch.where(active, n1, norm)
    u, dH = m.field(*x)
    return x[0] + h * u, x[1] - h * dH


def _accept(H0, H1, u):
    d = torch.nan_to_num(H0 - H1, nan=-math.inf)
    acc = torch.exp(d).clamp(max=1.0)
    return acc, u < acc


def _where(take, new, old):
    return tuple(torch.where(take.reshape((-1,) + (1,) * (a.dim() - 1)), a, b) for a, b in zip(new, old))


def _rmhmc(m, case, q, z, u):
    state, samples, accs = (q,) + m.logp_grad(q), [], []
    for t in range(case["T"]):
        p0 = m.draw(state[0], z[t])
        H0 = m.energy(state[0], p0)[0]
        q1, p1 = state[0], p0
        for _ in range(case["L"]):
            q1, p1 = _midpoint(m, q1, p1, case["eps"], case["iters"])
        H1, v1 = m.energy(q1, p1)
        acc, take = _accept(H0, H1, u[t])
        new = (q1,) + m.logp_grad(q1)
        state = _where(take, new, state)
        samples.append(state[0])
        accs.append(acc)
    return _answer(case, state, samples, accs, p0, H1, take, (q1, -p1, -v1, new[1]))


def _answer(case, state, samples, accs, draw, energy, take, end):
    if case["T"] > 1:
        return {"state": state, "samples": torch.stack(samples), "acceptance": torch.stack(accs)}
    return {"state": state, "draw": draw, "energy": energy, "acceptance": accs[0], "accepted": None, "end": end}


def _monge_half(alpha2, v, J, g, Hv, L, Hg, eps):
    """Half step of the Lagrangian integrator, unit mass, in the form the sampler
    uses by default (no alpha2 in the velocity's rank-one correction)."""
    dot = lambda a, b: (a * b).sum(1)  # noqa: E731
    d1 = 1 + 0.5 * eps * alpha2 * dot(Hv, g)
    J = J - torch.log(d1.abs())
    root = L.sqrt()[:, None]
    dphi = -g + alpha2 * Hg / root
    tmp = v - 0.5 * eps * root * (dphi - alpha2 * dot(dphi, g)[:, None] * g)
    v = tmp - (0.5 * eps * dot(tmp, Hv) / d1)[:, None] * g
    return v, J + torch.log((1 - 0.5 * eps * alpha2 * dot(Hg, v)).abs())


def _funnel_lmc(m, case, q, z, u):
    a2, eps = 1.0, case["eps"]

    def at(q):
        logp, g = m.logp_grad(q)
        L = 1 + a2 * (g * g).sum(1)
        gn = g / L.sqrt()[:, None]
        return logp, g, L, gn, m.hvp(q, gn) / L.sqrt()[:, None]

    def energy(logp, v, gn, L, J):
        return -logp - 0.5 * torch.log(L) + 0.5 * (v * v).sum(1) + 0.5 * L * a2 * (v * gn).sum(1) ** 2 - J

    logp, g = m.logp_grad(q)
    state, samples, accs = (q, logp, g, torch.zeros_like(logp)), [], []
    for t in range(case["T"]):
        q1, J = state[0], state[3]
        logp, g, L, gn, Hg = at(q1)
        inv = torch.eye(m.D, device=q.device, dtype=F64) - a2 * gn[:, :, None] * gn[:, None, :]
        v0 = v = (torch.linalg.cholesky(inv) @ z[t][..., None])[..., 0]
        H0 = energy(logp, v, gn, L, J)
        for _ in range(case["L"]):
            v, J = _monge_half(a2, v, J, gn, m.hvp(q1, v) / L.sqrt()[:, None], L, Hg, eps)
            q1 = q1 + eps * v
            logp, g, L, gn, Hg = at(q1)
            v, J = _monge_half(a2, v, J, gn, m.hvp(q1, v) / L.sqrt()[:, None], L, Hg, eps)
        H1 = energy(logp, v, gn, L, J)
        acc, take = _accept(H0, H1, u[t])
        momentum = v + (a2 * L * (v * g).sum(1))[:, None] * g
        state = _where(take, (q1, logp, g, J), state)
        samples.append(state[0])
        accs.append(acc)
    return _answer(case, state, samples, accs, v0, H1, take, (q1, -momentum, -v, logp))


def _lmc(m, case, q, z, u):
    eps = case["eps"]
    mv = lambda A, x: (A @ x[..., None])[..., 0]  # noqa: E731

    def half(geo, grad, v, J):
        s, lam, G, _, _, a = geo
        w = lam * (1 - 2 * s)
        omega = lambda v: 0.5 * m.gram(w * (v @ m.Xt))  # noqa: E731
        A = G + 0.5 * eps * omega(v)
        J = J - torch.linalg.slogdet(A)[1]
        v = torch.linalg.solve(A, mv(G, v) - 0.5 * eps * (0.5 * (w * a) @ m.X - grad))
        return v, J + torch.linalg.slogdet(G - 0.5 * eps * omega(v))[1]

    def energy(logp, geo, v, J):
        return -logp - torch.log(torch.diagonal(geo[3], dim1=1, dim2=2)).sum(1) + 0.5 * (v * mv(geo[2], v)).sum(1) - J

    logp, grad = m.logp_grad(q)
    J = torch.zeros_like(logp)
    old, geo = (q, logp, grad, J), m.geometry(q)
    v0 = v = torch.linalg.solve_triangular(geo[3].transpose(1, 2), z[0][..., None], upper=True)[..., 0]
    H0 = energy(logp, geo, v, J)
    for _ in range(case["L"]):
        v, J = half(geo, grad, v, J)
        q = q + eps * v
        geo = m.geometry(q)
        logp, grad = m.logp_grad(q)
        v, J = half(geo, grad, v, J)
    H1 = energy(logp, geo, v, J)
    acc, take = _accept(H0, H1, u[0])
    state = _where(take, (q, logp, grad, J), old)
    return _answer(case, state, None, [acc], v0, H1, take, (q, -mv(geo[2], v), -v, logp))


def _mmala(m, case, q, z, u):
    eps = case["eps"]
    mv = lambda A, x: (A @ x[..., None])[..., 0]  # noqa: E731

    def at(q):
        s, lam, G, _, Gi, a = m.geometry(q)
        logp, grad = m.logp_grad(q)
        gamma = -mv(Gi, (lam * (1 - 2 * s) * a) @ m.X)
        chol = torch.linalg.cholesky(2 * eps * Gi)
        return (q, logp, grad, G, gamma), q + eps * mv(Gi, grad) + eps * gamma, chol

    def logq(to, mean, chol):
        r = torch.linalg.solve_triangular(chol, (to - mean)[..., None], upper=False)[..., 0]
        return -0.5 * (r * r).sum(1) - torch.log(torch.diagonal(chol, dim1=1, dim2=2)).sum(1)

    state, samples, accs = at(q)[0], [], []
    for t in range(case["T"]):
        _, mean, chol = at(state[0])
        new, mean1, chol1 = at(mean + mv(chol, z[t]))
        weight = new[1] + logq(state[0], mean1, chol1) - state[1] - logq(new[0], mean, chol)
        acc, take = _accept(weight, torch.zeros_like(weight), u[t])
        state = _where(take, new, state)
        samples.append(state[0])
        accs.append(acc)
    if case["T"] > 1:
        return {"state": state, "samples": torch.stack(samples), "acceptance": torch.stack(accs)}
    return {"state": state, "proposal": new, "acceptance": accs[0], "accepted": None}


def _tangent_exact(m, case, q, z, u):
    """Forward-mode derivative in log(step size) of the executed computation."""
    import torch.autograd.forward_ad as fw

    with fw.dual_level():
        e = torch.tensor(case["eps"], device=q.device, dtype=F64)
        eps = fw.make_dual(e, e)
        p0 = m.draw(q, z[0])
        q1, p1 = q, p0
        for _ in range(case["L"]):
            q1, p1 = _midpoint(m, q1, p1, eps, case["iters"])
        acc = torch.exp(m.energy(q, p0)[0] - m.energy(q1, p1)[0]).clamp(max=1.0)
        sq = ((q1 - q) ** 2).sum(1)
        val = {k: fw.unpack_dual(t) for k, t in (("objective", acc * sq), ("acceptance", acc), ("sq_jump", sq))}
    d = lambda t: torch.stack([t.tangent, torch.zeros_like(t.tangent)], 1)  # noqa: E731
    return {"objective": val["objective"].primal, "acceptance": val["acceptance"].primal,
            "sq_jump": val["sq_jump"].primal, "d_objective": d(val["objective"]), "d_sq_jump": d(val["sq_jump"])}


def _ess(x):
    """Effective sample size (Geyer's initial monotone sequence over the mean
    autocovariance of the chains) and R-hat of x [T, C, D]."""
    T, C, _ = x.shape
    mean = x.mean(0)
    f = torch.fft.rfft(x - mean, n=2 * T, dim=0)
    acov = torch.fft.irfft(f * f.conj(), n=2 * T, dim=0)[:T].mean(1) / T
    var0 = acov[0] * T / (T - 1.0)
    total = acov[0] + mean.var(0)
    rho = 1 - (var0 - acov[:T - T % 2]) / total
    rho[0] = 1.0
    even, odd = rho[0::2].clone(), rho[1::2].clone()
    keep = torch.cumprod(((even + odd) > 0).to(F64), 0) > 0
    last = (keep.sum(0) - 1).clamp(min=0) + 1  # first pair left out (at least the second)
    pair = torch.arange(even.shape[0], device=x.device)[:, None]
    even = torch.where(torch.where(pair == last, even > 0, keep), even, 0.0)
    odd = torch.where(keep, odd, 0.0)
    pairs = even + odd
    low = torch.cummin(pairs, 0).values
    above = pairs > torch.cat([pairs[:1], low[:-1]])
    even, odd = torch.where(above, low / 2, even), torch.where(above, low / 2, odd)
    tau = -1 + 2 * (even + odd).sum(0) - torch.gather(even, 0, last.clamp(max=even.shape[0] - 1)[None])[0]
    within = x.var(0).mean(0)
    between = T * mean.var(0)
    return {"ess": T * C / tau.clamp(min=1 / math.log10(T * C)),
            "rhat": torch.sqrt((between / within + T - 1) / T)}


def _chunked(f, m, case, inp, rows):
    """f over chains in chunks that hold at most 2.5e8 values of [chains, N, D]."""
    q, z, u = inp["q"].to(F64)[rows], inp["z"].to(F64)[:, rows], inp["u"][:, rows]
    q, z = q[:, :m.D], z[:, :, :m.D]
    per = max(1, int(2.5e8 // (m.N * m.D)))
    parts = [f(m, case, q[i:i + per], z[:, i:i + per], u[:, i:i + per]) for i in range(0, q.shape[0], per)]
    return _joined(parts, case["T"] if "T" in case else 1)


def _joined(parts, T, width=None):
    """Per-chain results of several groups of chains in one; coordinates past a
    group's own are zero."""
    first = parts[0]
    if first is None:
        return None
    if isinstance(first, dict):
        return {k: _joined([p[k] for p in parts], 0 if k not in ("samples", "acceptance") or T == 1 else T, width)
                for k in first}
    if isinstance(first, tuple):
        return tuple(_joined(list(p), T, width) for p in zip(*parts))
    dim = 1 if T > 1 else 0
    if width is not None and first.dim() > dim + 1:
        parts = [torch.nn.functional.pad(p, (0, width - p.shape[-1])) for p in parts]
    return torch.cat(parts, dim)


def exact(case, seed):
    kind = case["kind"]
    if kind == "nuts":
        return None  # the tree is grown leaf by leaf and chain by chain: minutes in plain torch
    inp = _inputs(case, seed)
    if kind == "ess":
        r = _ess(inp["x"].to(F64))
        return {k: v.squeeze() for k, v in r.items()}
    if kind in ("funnel_rmhmc", "funnel_lmc"):
        f = _rmhmc if kind == "funnel_rmhmc" else _funnel_lmc
        return f(_Funnel(case["D"]), case, inp["q"].to(F64), inp["z"].to(F64), inp["u"])
    f = {"rmhmc": _rmhmc, "batch": _rmhmc, "lmc": _lmc, "mmala": _mmala, "tangent": _tangent_exact}[kind]
    if kind != "batch":
        X, y, _ = inp["data"][0]
        return _chunked(f, _Logistic(X, y), case, inp, slice(None))
    per = case["per"]
    parts = [_chunked(f, _Logistic(X, y), case, inp, slice(p * per, (p + 1) * per))
             for p, (X, y, _) in enumerate(inp["data"])]
    return _joined(parts, case["T"], inp["q"].shape[1])
