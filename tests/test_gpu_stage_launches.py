"""Two-phase steps at the phase sizes where the lanes per particle of the list
stages change, with partial workgroups, and with partner lists and windows
that hold every partner or overflow: two steps of one call (the first one's
final launch packs the second), against the oracle; and the split launches
that the profile times give the same numbers."""
import numpy as np
import pytest

import oracle
from helpers import crop_phase, field_errors
from sources_amd import abi, scenarios
from sources_amd.sph import Solver

pytestmark = pytest.mark.gpu

FIELDS = {"water": ("x", "vx", "rho", "p", "vof", "dvx", "av", "txx", "txy", "tyy"),
          "soil": ("x", "vx", "rho", "p", "vof", "sxx", "sxy", "syy", "dvx", "av")}


def _case(nw, ns, skf=1, nnps=1, vary_h=False, squeeze=1.0, perturb=False):
    # at least nw water and ns soil particles: tank 4 x 1.5, column 1 x 1 (dx: the unit)
    dx = min((2.1 / (nw + 400)) ** 0.5 * 0.1, (0.9 / (ns + 400)) ** 0.5 * 0.1)
    sc = scenarios.submerged_column(dx=dx, soil_w=0.1, soil_h=0.1, tank_w=0.2, tank_h=0.12, jitter=0.05, seed=nw + ns,
                                    skf=skf, max_interaction=0)
    sc.params.nnps = nnps
    assert sc.water.n >= nw and sc.soil.n >= ns, (sc.water.n, sc.soil.n)
    # (the leftmost of each phase: the soil column, its pore water and the wall)
    sc.water, sc.soil = (crop_phase(ph, np.sort(np.argsort(ph.x[:ph.n, 0], kind="stable")[:n]))
                         for ph, n in ((sc.water, nw), (sc.soil, ns)))
    r, ulp = np.random.default_rng(nw), np.random.default_rng(ns)
    for ph in (sc.water, sc.soil):
        ph.set_max_interaction(int(70 / squeeze ** 2) * ph.n + 4000)
        ph.vx[:] = r.uniform(-0.05, 0.05, ph.vx.shape) * (ph.itype[:, None] > 0)
        if vary_h:
            ph.hsml *= r.uniform(0.97, 1.03, ph.n)
        if squeeze < 1.0:   # a dense patch: more candidates than a list holds
            c = ph.x.mean(axis=0)
            near = (np.abs(ph.x - c).max(axis=1) < 8 * dx) & (ph.itype > 0)
            ph.x[near] = c + (ph.x[near] - c) * squeeze
        if perturb:
            ph.rho *= 1.0 + ulp.choice([-1.0, 1.0], ph.n) * 2.0 ** -52
    return sc


@pytest.mark.parametrize("kw", [
    dict(nw=321, ns=257), dict(nw=4096, ns=193), dict(nw=4097, ns=97), dict(nw=20000, ns=4096),
    dict(nw=20001, ns=4097), dict(nw=2000, ns=1500, vary_h=True), dict(nw=2000, ns=1500, nnps=2),
    dict(nw=3000, ns=2000, squeeze=0.5), dict(nw=21000, ns=5000, squeeze=0.5),
    dict(nw=12000, ns=600, skf=2), dict(nw=12001, ns=600, skf=3), dict(nw=3000, ns=2000, skf=3, squeeze=0.6)],
    ids=lambda k: "-".join(f"{a}{b}" for a, b in k.items()))
def test_two_steps_match_the_oracle(kw):
    print(kw, flush=True)
    sc = _case(**kw)
    s = Solver(sc.params, sc.water, sc.soil)
    s.time_integration(2, sync=True)
    s.close()
    ref, near = _case(**kw), _case(perturb=True, **kw)
    for c in (ref, near):
        oracle.time_integration(c.params, c.water, c.soil, 0, 2)
    bad = {}
    for name, f in FIELDS.items():
        errs = field_errors(getattr(sc, name), getattr(ref, name), f)
        sens = field_errors(getattr(near, name), getattr(ref, name), f)
        # within 1e-12 norm-wise, or within 16x the oracle's own change under
        # a one-ulp change of its input densities
        bad.update({(name, k): (errs[k], sens[k]) for k in f if not errs[k] <= max(1e-12, 16.0 * sens[k])})
    assert not bad, bad


@pytest.mark.parametrize("precision", [abi.SPHG_FP64, abi.SPHG_MIXED], ids=["fp64", "mixed"])
def test_merged_and_split_launches_agree(precision):
    out = []
    for prof in (False, True):
        sc = _case(nw=6000, ns=3000)
        sc.params.precision = precision
        s = Solver(sc.params, sc.water, sc.soil)
        s.profile(prof)
        s.time_integration(5, sync=True)
        s.close()
        out.append(sc)
    # the same device code on the same operands
    for name, fields in FIELDS.items():
        for f in fields:
            np.testing.assert_array_equal(getattr(getattr(out[0], name), f), getattr(getattr(out[1], name), f), f)
