"""GPU parity of the float64 logistic passes at the edges of their tiles.

The passes take rows in blocks of 16 dealt to four waves and features in tiles
of 16 (one to four up to 64 features, six or eight up to 128), with whole
last tiles loaded as pairs; these sizes sit on, just below and just above
every one of those limits.  One RMHMC transition (Gram with and without the
likelihood, inverse, quadratic forms) and one LMC transition (weighted Grams,
G v) against the float64 oracle.  Tolerance 1e-10 norm-wise relative, as in
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
from geomjax_amd.synthetic import make_logistic
from oracle import lmcmc as olc
from oracle import models as om
from oracle import rmhmc as orm
from tests.helpers import rel_err, seeded_normal, seeded_uniform

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
SIZES = [(1, 1), (1, 3), (15, 2), (16, 15), (17, 16), (63, 17), (64, 32), (65, 33), (130, 47), (100, 48), (129, 49),
         (90, 63), (113, 64)]
WIDE = [(70, 65), (97, 96), (130, 97), (144, 127)]


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
