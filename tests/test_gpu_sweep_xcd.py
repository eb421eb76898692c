"""GPU: a sweep on one XCD (small lattices, the default there), the sweep over
all XCDs and the colour passes give the same run bit for bit, on both sides of
the line between them (100 tiles a colour and layer), for the smallest lattice,
films that start across two tile layers, short and long windows."""
import numpy as np
import pytest

from mulskips_amd import models
from mulskips_amd.engine import Engine

pytestmark = pytest.mark.gpu

CASES = {  # box, tile, slab, policy, k, events
    "smallest": ("si", (96, 96, 130), 48, 45, 0, 1.0, 1500),
    "two_layers": ("sige", (96, 96, 150), 16, 48, 1, 2.0, 4000),
    "line": ("sige", (480, 480, 130), 24, 45, 1, 2.0, 20000),
    "above_line": ("sige", (528, 480, 130), 24, 48, 0, 0.0, 3000),
    "sic": ("sic", (192, 144, 200), 24, 96, 1, 4.0, 20000),
}


def _engine(name):
    model, box, tile, slab, policy, k, events = CASES[name]
    tables = {"si": models.si_c1_tables, "sic": models.sic_c2_tables,
              "sige": lambda: models.sige_alloy_tables(1200.0, 1.0, 0.3)}[model]()
    e = Engine(box, tables, seed=7, tile=tile, tau_policy=policy, events_per_pass=k, frozen_below_z=slab - 11)
    if model == "sige":
        e.build_alloy_slab(slab, 0.3)
    else:
        e.build_slab(1 if model == "sic" else 0, slab)
    return e, events


@pytest.mark.parametrize("name", CASES)
def test_the_three_sweeps_agree(name):
    out = {}
    for schedule in ("colours", "tiles", None):
        e, events = _engine(name)
        if schedule:
            e.set_schedule(schedule)
        runs = [e.run(events), e.run(events // 3)]
        lat, mc, bulk, void = e.store_state()
        out[schedule] = (runs, lat, mc, e.counters()[0], e.diagnostics())
        e.close()
    want = out["colours"]
    assert want[0][0][0] >= CASES[name][-1]
    for schedule in ("tiles", None):
        got = out[schedule]
        assert got[0] == want[0] and got[4] == want[4], schedule
        assert np.array_equal(got[1], want[1]) and np.array_equal(got[3], want[3])
        for k in want[2]:
            assert np.array_equal(got[2][k], want[2][k]), k
