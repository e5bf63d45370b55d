"""Single-phase soil at the particle counts where the number of lanes per
particle changes, and at counts that leave partial waves: three steps of one
call (the later ones start from the cell keys the pass before left), against
the oracle."""
import numpy as np
import pytest

import oracle
from helpers import crop_phase, field_errors
from sources_amd import scenarios
from sources_amd.sph import Solver

pytestmark = pytest.mark.gpu

FIELDS = ("x", "vx", "rho", "p", "sxx", "sxy", "syy", "dvx", "av", "txx", "txy", "tyy")


def _case(n, nnps, skf=1, vary_h=False, density=False, perturb=False):
    dx = (0.0045 / (n + 400)) ** 0.5
    sc = scenarios.soil_collapse(dx=dx, width=0.1, height=0.05, skf=skf, jitter=0.1, seed=n, max_interaction=0)
    sc.params.nnps = nnps
    sc.params.dt = min(1.0e-5, 0.05 * dx / sc.params.soil_c)
    if density:
        sc.params.summation_density = 1
    assert sc.soil.n >= n, sc.soil.n
    sc.soil = crop_phase(sc.soil, np.sort(np.argsort(sc.soil.x[:sc.soil.n, 0], kind="stable")[:n]))
    sc.soil.set_max_interaction(40 * n + 400)
    r = np.random.default_rng(n)
    sc.soil.vx[:] = r.uniform(-0.05, 0.05, sc.soil.vx.shape) * (sc.soil.itype[:, None] > 0)
    if vary_h:
        sc.soil.hsml *= r.uniform(0.97, 1.03, n)
    if perturb:
        sc.soil.rho *= 1.0 + np.random.default_rng(n + 1).choice([-1.0, 1.0], n) * 2.0 ** -52
    return sc


@pytest.mark.parametrize("kw", [
    dict(n=1, nnps=1), dict(n=65, nnps=1), dict(n=1037, nnps=2, skf=3), dict(n=9999, nnps=2, density=True),
    dict(n=10000, nnps=2), dict(n=10001, nnps=2), dict(n=12000, nnps=1, vary_h=True), dict(n=40000, nnps=2),
    dict(n=40001, nnps=2, skf=4), dict(n=80000, nnps=2), dict(n=80001, nnps=2)],
    ids=lambda k: "-".join(f"{a}{b}" for a, b in k.items()))
def test_three_steps_match_the_oracle(kw):
    print(kw, flush=True)
    sc = _case(**kw)
    s = Solver(sc.params, None, sc.soil)
    s.time_integration(3, sync=True)
    s.close()
    ref, near = _case(**kw), _case(perturb=True, **kw)
    for c in (ref, near):
        oracle.time_integration(c.params, None, c.soil, 0, 3)
    errs, sens = field_errors(sc.soil, ref.soil, FIELDS), field_errors(near.soil, ref.soil, FIELDS)
    # within 1e-12 norm-wise, or within 16x the oracle's own change under a
    # one-ulp change of its input density
    bad = {f: (errs[f], sens[f]) for f in FIELDS if not errs[f] <= max(1e-12, 16.0 * sens[f])}
    assert not bad, bad
