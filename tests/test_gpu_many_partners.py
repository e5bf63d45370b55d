"""Particles with more partners than the fast forms hold: graph nodes of more
neighbours than a wavefront keeps edge operands for in the backward pass (28), and
single-phase water with more candidates than a 128-bit mask (its rows are walked)."""
import numpy as np
import pytest

import gnn_ref as G
import oracle
from helpers import field_errors
from sources_amd import scenarios
from sources_amd.sph import Solver
from sources_amd.surrogate import Surrogate
from test_gpu_single_water import FIELDS, _case

pytestmark = pytest.mark.gpu

# as for the gradients of nodes of few neighbours: BF16 operands rounded as in the
# reference, FP32 against FP64 partial sums at a rounding boundary; the pairs of
# slots past the 28th are a tenth of all edges and more
TOL = 3e-4


def off(a, b):
    return np.linalg.norm(np.asarray(a, np.float64) - b) / np.linalg.norm(b)


@pytest.mark.parametrize("scale", [1.4, 1.6])   # up to about 36 and 44 neighbours (48 fit)
def test_gradients_of_nodes_with_many_neighbours(scale):
    print("scale", scale, flush=True)
    sc = scenarios.submerged_column(dx=0.0071, soil_w=0.1, soil_h=0.05, tank_w=0.3, tank_h=0.12, jitter=0.02, seed=7)
    for p in (sc.water, sc.soil):
        p.hsml *= scale
    s = Solver(sc.params, sc.water, sc.soil)
    s.time_integration(2, sync=False)
    g = Surrogate(s, ksteps=2, max_samples=1, seed=3)
    g.record(1)
    d = g.debug(0)
    assert 28 < d["nd"].max() <= 48 and d["nd"].min() < 28
    n = len(d["nd"])
    ii, jj = G.edges(d["nb"], d["nd"])
    e = G.edge_features(d["raw"], ii, jj)
    tgt = d["tgt"].astype(np.float64) / d["out_scale"][None, :].astype(np.float64)
    L, grad, y = G.loss_and_grad(g.weights().astype(np.float64), d["nf"], e, ii, n, tgt, d["tw"].astype(np.float64),
                                 rb=True)
    assert off(d["y"], y) <= TOL
    assert abs(d["loss"] - L) <= TOL * L
    for a, b in ((G.O_W1, G.O_W2), (G.O_W2, G.O_W3), (G.O_W3, G.O_B3), (G.O_B3, G.O_W4), (G.O_W4, G.O_B4),
                 (G.O_B4, G.O_W5), (G.O_W5, G.O_B5), (G.O_B5, G.NPARAM)):
        assert off(d["grad"][a:b], grad[a:b]) <= TOL, (a, b)
    g.close()
    s.close()


def _crowded(n, skf, scheme, perturb=False):
    sc = _case(n, 1, scheme, False, perturb)
    sc.params.skf = skf
    sc.water.hsml *= 1.25   # (radius 3h: 9 cells of 4.5 x 4.5 particles)
    sc.water.set_max_interaction(60 * n)
    return sc


@pytest.mark.parametrize("n,skf,scheme", [(65, 3, 1), (2051, 3, 1), (2051, 2, 2), (20500, 3, 2)])
def test_water_with_more_candidates_than_a_mask(n, skf, scheme):
    print("particles", n, flush=True)
    sc = _crowded(n, skf, scheme)
    s = Solver(sc.params, sc.water)
    s.time_integration(2, sync=True)
    s.close()
    ref, near = _crowded(n, skf, scheme), _crowded(n, skf, scheme, perturb=True)
    for c in (ref, near):
        oracle.time_integration(c.params, c.water, None, 0, 2)
    errs, sens = field_errors(sc.water, ref.water, FIELDS), field_errors(near.water, ref.water, FIELDS)
    # within 1e-12 norm-wise, or within 16x the oracle's own change under a
    # one-ulp change of its input density
    bad = {f: (errs[f], sens[f]) for f in FIELDS if not errs[f] <= max(1e-12, 16.0 * sens[f])}
    assert not bad, bad
