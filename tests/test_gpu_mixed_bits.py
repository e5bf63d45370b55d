"""The FP32 pair terms of mixed precision, bit for bit: a trajectory in FP32 terms
parts for good at the first flipped rounding, so these do not depend on how a
kernel visits its partners (windows, masks, rows) or on the phase's size.  CRC-32
words over all fields of a phase after three steps, recorded from the kernels that
gathered partners through 128-bit masks: particles with few candidates, crowded
ones (the radius-3h kernels, a squeezed patch) and varying smoothing lengths."""
import zlib

import numpy as np
import pytest

from sources_amd import abi
from sources_amd.sph import Solver
from test_gpu_learned_steps import FIELDS, MASK
from test_gpu_stage_launches import _case

pytestmark = pytest.mark.gpu

# (case, neighbour lists, word of the water, of the soil)
PINNED = [
    (dict(nw=321, ns=257), "1", 0xf66d3b06, 0x924c7052),
    (dict(nw=20001, ns=4097), "1", 0x24240cbd, 0xf4e69c44),
    (dict(nw=4097, ns=1025), "0", 0x5b6890d3, 0xf0717575),
    (dict(nw=3000, ns=2000, squeeze=0.5), "1", 0x1b6aea84, 0x287dfdf2),
    (dict(nw=3000, ns=2000, squeeze=0.5), "0", 0xcec18553, 0x0f0539a9),
    (dict(nw=3000, ns=2600, skf=2), "1", 0x16df656c, 0x235393e0),
    (dict(nw=12001, ns=2600, skf=3), "1", 0xb6e2bbbf, 0xb511b4a0),
    (dict(nw=3000, ns=2600, skf=3), "0", 0x36248c66, 0x2a93540c),
    (dict(nw=3000, ns=2600, skf=4, squeeze=0.5), "1", 0x7dfecde3, 0x26227cfe),
    (dict(nw=2000, ns=1500, vary_h=True), "1", 0x12b73c93, 0x3aedec5d),
]


def words(kw):
    sc = _case(**kw)
    sc.params.precision = abi.SPHG_MIXED
    s = Solver(sc.params, sc.water, sc.soil)
    s.time_integration(3, sync=False)
    out = []
    for name in ("water", "soil"):
        s.sync(name, MASK)
        crc = 0
        for f in FIELDS:
            crc = zlib.crc32(np.ascontiguousarray(getattr(getattr(sc, name), f)).tobytes(), crc)
        out.append(crc)
    s.close()
    return out


@pytest.mark.parametrize("kw,lists,water,soil", PINNED,
                         ids=lambda v: "-".join(f"{a}{b}" for a, b in v.items()) if isinstance(v, dict) else None)
def test_mixed_steps_keep_their_bits(kw, lists, water, soil, monkeypatch):
    print(kw, lists, flush=True)
    monkeypatch.setenv("SPHG_NLIST", lists)
    assert [hex(v) for v in words(kw)] == [hex(water), hex(soil)]
