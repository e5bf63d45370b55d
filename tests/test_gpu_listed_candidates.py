"""Listed candidates outside the support (in the lists' skin) count nothing: a
particle that is not finite spoils its partners alone, and a wall particle
within r0 but beyond the support repels nothing.  One step against the oracle,
whose pairs are those within the support, at the phase sizes where the lanes per
particle change."""
import numpy as np
import pytest

import oracle
from helpers import field_errors
from sources_amd import abi
from sources_amd.sph import Solver
from test_gpu_stage_launches import _case

pytestmark = pytest.mark.gpu

SIZES = [dict(nw=321, ns=257), dict(nw=4097, ns=1025), dict(nw=20001, ns=4097)]


@pytest.mark.parametrize("precision", [abi.SPHG_FP64, abi.SPHG_MIXED], ids=["fp64", "mixed"])
@pytest.mark.parametrize("value", [np.nan, np.inf], ids=str)
@pytest.mark.parametrize("kw", SIZES, ids=lambda k: str(k["nw"]))
def test_a_wall_particle_that_is_not_finite(kw, value, precision):
    sc, ref = _case(**kw), _case(**kw)
    sc.params.precision = precision
    r = np.random.default_rng(1)
    for c in (sc, ref):
        for ph in (c.water, c.soil):
            ph.hsml *= 1.1   # (support 2.64 dx, lists to 2.9 dx: the lattice's 2.83 dx between them)
            # (its velocity: it stays where it is; beside real particles)
            wall = np.flatnonzero(ph.itype[:ph.n] < 0)
            real = ph.x[:ph.n][ph.itype[:ph.n] > 0]
            near = [i for i in wall if np.min(np.hypot(*(real - ph.x[i]).T)) < 1.5 * ph.hsml[0]]
            ph.vx[near[len(near) // 2]] = value
    s = Solver(sc.params, sc.water, sc.soil)
    s.time_integration(1, sync=True)
    s.close()
    oracle.time_integration(ref.params, ref.water, ref.soil, 0, 1)
    for name in ("water", "soil"):
        got, want = ({f: ~np.isfinite(getattr(getattr(c, name), f)) for f in ("drho", "dvx")} for c in (sc, ref))
        assert want["drho"].sum() > 3   # (it has partners)
        for f in want:
            np.testing.assert_array_equal(got[f], want[f], f"{name} {f}")


@pytest.mark.parametrize("precision,tol", [(abi.SPHG_FP64, 1e-12), (abi.SPHG_MIXED, 2e-3)], ids=["fp64", "mixed"])
@pytest.mark.parametrize("kw", SIZES, ids=lambda k: str(k["nw"]))
def test_repulsion_ends_at_the_support(kw, precision, tol):
    sc, ref = _case(**kw), _case(**kw)
    sc.params.precision = precision
    for c in (sc, ref):
        c.params.p1, c.params.p2 = 2.0, 1.0
        for ph in (c.water, c.soil):
            ph.hsml *= 1.1   # (as above)
            ph.dspp = 3.0 * ph.hsml[0]
    s = Solver(sc.params, sc.water, sc.soil)
    s.time_integration(1, sync=True)
    s.close()
    oracle.time_integration(ref.params, ref.water, ref.soil, 0, 1)
    for name in ("water", "soil"):
        e = field_errors(getattr(sc, name), getattr(ref, name), ("dvx",))
        assert e["dvx"] <= tol, (name, e)
