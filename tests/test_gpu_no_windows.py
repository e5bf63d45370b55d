"""The forms of the two-phase step whose partners are not read from LDS windows
(smoothing lengths that vary, link_list's reach, no neighbour lists,
Mohr-Coulomb or other than integer repulsion exponents), at the phase sizes
where the lanes per particle change, with candidate masks that hold every
candidate, take a second round or overflow: two steps of one call against the
oracle, and batches of such contexts against the same contexts alone."""
import numpy as np
import pytest

import oracle
from helpers import field_errors
from sources_amd import abi
from sources_amd.batch import Batch
from sources_amd.sph import Solver
from test_gpu_batch import FIELDS as BATCH_FIELDS
from test_gpu_batch import cases
from test_gpu_stage_launches import FIELDS, _case

pytestmark = pytest.mark.gpu

SMALL, TWO, ONE = dict(nw=321, ns=257), dict(nw=4097, ns=1025), dict(nw=20001, ns=4097)


@pytest.mark.parametrize("kw,params,lists", [
    (dict(SMALL, vary_h=True), {}, "1"), (dict(TWO, vary_h=True), {}, "1"), (dict(ONE, vary_h=True), {}, "1"),
    (SMALL, {}, "0"), (TWO, {}, "0"), (ONE, {}, "0"), (dict(TWO, vary_h=True), {}, "0"),
    (dict(SMALL, nnps=2), {}, "0"), (dict(ONE, nnps=2), {}, "1"),
    (dict(nw=3000, ns=2000, skf=3), {}, "0"), (dict(nw=13000, ns=600, skf=2), {}, "0"),
    (dict(nw=3000, ns=2000, skf=2, vary_h=True), {}, "1"), (dict(nw=3000, ns=2000, squeeze=0.5), {}, "0"),
    (dict(nw=21000, ns=5000, squeeze=0.5, vary_h=True), {}, "1"),
    (TWO, dict(yield_criterion=1), "1"), (dict(ONE, vary_h=True), dict(yield_criterion=1), "0"),
    (TWO, dict(p1=11.5), "1"), (ONE, dict(p1=11.5, p2=3.5), "0")],
    ids=lambda v: "-".join(f"{a}{b}" for a, b in v.items()) if isinstance(v, dict) else "lists" + v)
def test_two_steps_match_the_oracle(kw, params, lists, monkeypatch):
    print(kw, params, lists, flush=True)
    monkeypatch.setenv("SPHG_NLIST", lists)

    def make(**more):
        sc = _case(**kw, **more)
        for k, v in params.items():
            setattr(sc.params, k, v)
        return sc

    sc, ref, near = make(), make(), make(perturb=True)
    s = Solver(sc.params, sc.water, sc.soil)
    s.time_integration(2, sync=True)
    s.close()
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


@pytest.mark.parametrize("precision,nnps,vary_h,lists", [
    (abi.SPHG_FP64, 2, False, "1"), (abi.SPHG_FP64, 1, False, "0"), (abi.SPHG_FP64, 1, True, "1"),
    (abi.SPHG_MIXED, 1, False, "0"), (abi.SPHG_MIXED, 1, True, "1")])
def test_batch_is_bit_identical_to_solo(precision, nnps, vary_h, lists, monkeypatch):
    monkeypatch.setenv("SPHG_NLIST", lists)
    solo, bat = cases()[:2], cases()[:2]
    for c in solo + bat:
        c.params.precision, c.params.nnps = precision, nnps
        if vary_h:
            for ph in (c.water, c.soil):
                ph.hsml *= np.random.default_rng(3).uniform(0.98, 1.02, ph.hsml.shape)
    ss, sb = ([Solver(c.params, c.water, c.soil) for c in cs] for cs in (solo, bat))
    for s in ss:
        s.time_integration(140, sync=True)
    b = Batch(sb)
    b.run(140)
    assert b.staged
    for s in sb:
        s.sync_all()
    for a, c in zip(solo, bat):
        for ph in ("water", "soil"):
            for f in BATCH_FIELDS:
                if hasattr(getattr(a, ph), f):
                    np.testing.assert_array_equal(getattr(getattr(a, ph), f), getattr(getattr(c, ph), f), f)
    b.close()
    for s in ss + sb:
        s.close()
