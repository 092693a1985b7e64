"""GPU parity of the float64 logistic passes at the edges of their tiles.

The passes take rows in blocks of 16 dealt to four waves and features in tiles
of 16 (one to four up to 64 features, five to eight up to 128), with whole
last tiles loaded as pairs; these sizes sit on, just below and just above
every one of those limits.  One RMHMC transition (Gram with and without the
likelihood, inverse, quadratic forms) and one LMC transition (weighted Grams,
G v) against the float64 oracle.  What lies past a posterior's rows must not
matter: the same posterior before one whose rows are all NaN (the batch's rows
share one buffer) has to give its own results to the last bit.  Tolerance 1e-10 norm-wise relative, as in
the other float64 parity tests: rounding of order 1e-16 times the metric's
condition number (at most 1e4 here: its eigenvalues lie between the prior's
1e-2 and N / 4 D + 1e-2).
"""
import functools

import pytest
import torch

import geomjax_amd as gj
from geomjax_amd import random as gr
from geomjax_amd.rmhmc import implicit_midpoint
from geomjax_amd.rmhmc import sample as rmhmc_sample
from geomjax_amd.synthetic import make_logistic
from oracle import lmcmc as olc
from oracle import models as om
from oracle import rmhmc as orm
from tests.helpers import rel_err, seeded_normal, seeded_uniform

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
SIZES = [(1, 1), (1, 3), (15, 2), (16, 15), (17, 16), (63, 17), (64, 32), (65, 33), (130, 47), (100, 48), (129, 49),
         (90, 63), (113, 64)]
WIDE = [(70, 65), (65, 79), (33, 80), (90, 81), (97, 96), (130, 97), (81, 111), (64, 112), (113, 113), (144, 127),
        (40, 128)]


@pytest.mark.parametrize("N,D", SIZES + WIDE)
def test_rmhmc_step_at_tile_edges(N, D):
    print(f"case N={N} D={D}", flush=True)
    X, y, _ = make_logistic(N, D, 1000 + N + D)
    M = om.LogisticRegression(X, y, 100.0)
    q0, z, u = 0.5 * seeded_normal(N, 2, D), seeded_normal(D, 2, D), 0.0 * seeded_uniform(3, 2)
    so = orm.init(q0, M.logp)
    so1, io = orm.build_kernel(max_iters=3)((z, u), so, M.logp, 0.05, M.fisher_metric_fn, 1)
    model = gj.LogisticRegression(X, y, 100.0)
    s = gj.rmhmc.init(q0.to(DEV), model)
    assert rel_err(s.logdensity, so.logdensity) < 1e-12
    assert rel_err(s.logdensity_grad, so.logdensity_grad) < 1e-12
    alg = gj.rmhmc(model, 0.05, gj.FisherMetric(), 1,
                   integrator=functools.partial(implicit_midpoint, max_iters=3))
    s1, info = alg.step(gr.HostNoise(z.to(DEV), u.to(DEV)), s)
    ps, pso = info.proposal.state, io.proposal.state
    for name in ("position", "momentum", "velocity", "logdensity", "logdensity_grad"):
        assert rel_err(getattr(ps, name), getattr(pso, name)) < 1e-10, name
    assert rel_err(info.momentum, io.momentum) < 1e-10
    assert rel_err(info.energy, io.energy) < 1e-10
    assert rel_err(s1.position, so1.position) < 1e-10


@pytest.mark.parametrize("N,D", SIZES)
def test_lmc_step_at_tile_edges(N, D):
    print(f"case N={N} D={D}", flush=True)
    X, y, _ = make_logistic(N, D, 2000 + N + D)
    M = om.LogisticRegression(X, y, 100.0)
    q0, z, u = 0.5 * seeded_normal(N, 2, D), seeded_normal(D, 2, D), 0.0 * seeded_uniform(3, 2)
    so = olc.init(q0, M.logp)
    _, io = olc.build_kernel()((z, u), so, M.logp, 0.05, M.fisher_metric_fn, 1)
    model = gj.LogisticRegression(X, y, 100.0)
    s = gj.lmc.init(q0.to(DEV), model)
    _, info = gj.lmc(model, 0.05, gj.FisherMetric(), 1).step(gr.HostNoise(z.to(DEV), u.to(DEV)), s)
    ps, pso = info.proposal.state, io.proposal.state
    for name in ("position", "momentum", "velocity", "logdensity", "logdensity_grad"):
        assert rel_err(getattr(ps, name), getattr(pso, name)) < 1e-10, name
    assert (ps.volume_adjustment.cpu() - pso.volume_adjustment).abs().max().item() < 1e-10


@pytest.mark.parametrize("N,D", [(17, 5), (33, 47), (50, 63), (81, 65), (66, 72), (35, 79), (47, 80), (83, 97),
                                 (50, 104), (97, 111), (34, 112), (31, 127)])
def test_rows_past_the_posterior_do_not_matter(N, D):
    print(f"case N={N} D={D}", flush=True)
    X, y, _ = make_logistic(N, D, 3000 + N + D)
    alone = gj.LogisticRegression(X, y, 100.0)
    nan = gj.LogisticRegression(torch.full((N, D), float("nan")), torch.full((N,), float("nan")), 100.0)
    batch = gj.LogisticBatch([alone, nan], 2)
    q0, z, u = 0.5 * seeded_normal(N, 4, D), seeded_normal(D, 4, D), 0.5 * seeded_uniform(3, 4)
    integ = functools.partial(implicit_midpoint, max_iters=3)

    def both(run, first):
        return run(alone, slice(0, 2)), first(run(batch, slice(0, 4)))

    # value and gradient: float32 positions go through the float64 kernel too
    for dtype in (torch.float64, torch.float32):
        a, b = both(lambda m, c: m.value_and_grad(q0[c].to(DEV, dtype)), lambda r: tuple(v[:2] for v in r))
        assert bool(torch.isfinite(a[0]).all()) and bool(torch.isfinite(a[1]).all())
        assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])

    def step(m, c):
        alg = gj.rmhmc(m, 0.05, gj.FisherMetric(), 2, integrator=integ)
        s, info = alg.step(gr.HostNoise(z[c].to(DEV), u[c].to(DEV)), gj.rmhmc.init(q0[c].to(DEV), m))
        ps = info.proposal.state
        return s.position, s.logdensity, info.momentum, info.energy, ps.position, ps.momentum

    def sample(m, c):
        r = rmhmc_sample(gr.HostNoise(z[None, c].to(DEV), u[None, c].to(DEV)), gj.rmhmc.init(q0[c].to(DEV), m), m,
                         0.05, gj.FisherMetric(), 2, 1, integrator=integ)
        return r.state.position, r.state.logdensity, r.state.logdensity_grad

    for run in (step, sample):
        a, b = both(run, lambda r: tuple(v[:2] for v in r))
        for i, (v, w) in enumerate(zip(a, b)):
            assert bool(torch.isfinite(v).all()) and torch.equal(v, w), (run.__name__, i)
