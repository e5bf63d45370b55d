"""Single-phase water at the particle counts where the number of lanes per
particle changes, and at counts that leave partial waves: two steps of one
call (the second starts from the keys and half-step levels the first one's
force pass left), against the oracle."""
import numpy as np
import pytest

import oracle
from helpers import crop_phase, field_errors
from sources_amd import scenarios
from sources_amd.sph import Solver

pytestmark = pytest.mark.gpu

FIELDS = ("x", "vx", "rho", "p", "dvx", "av", "txx", "txy", "tyy")


def _case(n, nnps, scheme, vary_h, perturb=False):
    sc = scenarios.dam_break(dx=0.125 ** 0.5 / (1.1 * n + 100) ** 0.5, skf=1 if scheme == 1 else 4, jitter=0.2, seed=n,
                             max_interaction=0)
    sc.params.nnps = nnps
    sc.params.integrate_scheme = scheme
    sc.water = crop_phase(sc.water, np.arange(n))
    sc.water.set_max_interaction(40 * n)
    r = np.random.default_rng(n)
    sc.water.vx[:] = r.uniform(-0.5, 0.5, sc.water.vx.shape) * (sc.water.itype[:, None] > 0)
    if vary_h:
        sc.water.hsml *= r.uniform(0.97, 1.03, n)
    if perturb:
        sc.water.rho *= 1.0 + r.choice([-1.0, 1.0], n) * 2.0 ** -52
    return sc


@pytest.mark.parametrize("n,nnps,scheme,vary_h", [
    (1, 1, 1, False), (63, 1, 2, False), (65, 1, 1, True), (1037, 2, 2, False),
    (16384, 2, 1, False), (16385, 2, 2, False), (16500, 2, 1, True),
    (65536, 2, 1, False), (65537, 2, 2, False), (122880, 2, 2, False), (122881, 2, 1, False)])
def test_two_steps_match_the_oracle(n, nnps, scheme, vary_h):
    print("particles", n, flush=True)
    sc = _case(n, nnps, scheme, vary_h)
    s = Solver(sc.params, sc.water)
    s.time_integration(2, sync=True)
    s.close()
    ref, near = _case(n, nnps, scheme, vary_h), _case(n, nnps, scheme, vary_h, perturb=True)
    for c in (ref, near):
        oracle.time_integration(c.params, c.water, None, 0, 2)
    errs, sens = field_errors(sc.water, ref.water, FIELDS), field_errors(near.water, ref.water, FIELDS)
    # within 1e-12 norm-wise, or within 16x the oracle's own change under a
    # one-ulp change of its input density
    bad = {f: (errs[f], sens[f]) for f in FIELDS if not errs[f] <= max(1e-12, 16.0 * sens[f])}
    assert not bad, bad
