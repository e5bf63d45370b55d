"""Mixed precision at the phase sizes where the lanes per particle change, with
partial workgroups, lists and windows that hold every partner or overflow, and
smoothing lengths that vary (no windows): the rates of two steps against the
FP64 step of the same state, which the oracle pins."""
import pytest

from helpers import field_errors
from sources_amd import abi
from sources_amd.sph import Solver
from test_gpu_stage_launches import _case

pytestmark = pytest.mark.gpu

# FP32 pair terms of FP32 records: the bounds of the one-step comparison of
# the two precisions (2e-3 of the largest rate).  One partner lost or counted
# twice is a few percent of a sum of twenty.
RATE_TOL = 2e-3
RATES = {"water": ("drho", "dvx", "dvof"), "soil": ("drho", "dvx", "dsxx", "dsxy", "dsyy", "dp")}


@pytest.mark.parametrize("kw", [
    dict(nw=321, ns=257), dict(nw=4096, ns=193), dict(nw=4097, ns=97), dict(nw=20000, ns=4096),
    dict(nw=20001, ns=4097), dict(nw=2000, ns=1500, vary_h=True), dict(nw=3000, ns=2000, squeeze=0.5),
    dict(nw=21000, ns=5000, squeeze=0.5), dict(nw=12000, ns=600, skf=2), dict(nw=12001, ns=600, skf=3),
    dict(nw=5000, ns=4000, skf=4)],
    ids=lambda k: "-".join(f"{a}{b}" for a, b in k.items()))
def test_rates_match_fp64(kw):
    print(kw, flush=True)
    out = []
    for precision in (abi.SPHG_MIXED, abi.SPHG_FP64):
        sc = _case(**kw)
        sc.params.precision = precision
        s = Solver(sc.params, sc.water, sc.soil)
        s.time_integration(2, sync=True)
        s.close()
        out.append(sc)
    bad = {}
    for name, f in RATES.items():
        e = field_errors(getattr(out[0], name), getattr(out[1], name), f)
        bad.update({(name, k): v for k, v in e.items() if not v <= RATE_TOL})
    assert not bad, bad
