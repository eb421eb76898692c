"""GPU: the scheduled sweep over all XCDs, which "tiles" takes with more than
100 tiles a colour and layer, in each of its instances (second-neighbour term,
coverage species, laser annealing): the same state, lists, counters and clock as
the colour passes bit for bit, also where the schedule changes between runs, and
its event log replays serially through the oracle.  (The boxes of the other
schedule tests are small enough for the sweep on one XCD, but for one.)"""
import numpy as np
import pytest

from mulskips_amd import models
from mulskips_amd.engine import Engine
from oracle.oracle import Oracle
from tests.helpers import list_map, oracle_state, parity_mask, small_deck

pytestmark = pytest.mark.gpu

F2 = np.exp(-np.arange(13) * 0.05 / (8.617333262e-5 * 1600.0))
ONE_XCD = 100  # tiles a colour and layer that the sweep on one XCD takes at most
# name: (deck, builder mode, box, slab, tile, k, second-neighbour factors)
CASES = {
    "SiC-f2": ("surface", 1, (528, 480, 150), 96, 24, 4.0, F2),
    "CVD": ("CVD-Si-SiH2", 0, (384, 288, 192), 72, 16, 4.0, None),
    "Si": ("Si-SL", 0, (384, 288, 144), 72, 16, 1.0, None),
    "LA": (None, None, (384, 288, 192), 96, 16, 4.0, None),
}


def make(tmp_path, case, schedule):
    deck, mode, box, slab, tile, k, f2 = CASES[case]
    assert (box[0] // tile) * (box[1] // tile) // 4 > ONE_XCD
    if deck is None:
        tab, _ = models.la_sige_tables(2026)
        e = Engine(box, tab, seed=29, tile=tile, tau_policy=1, events_per_pass=k, la=models.LA_CONSTANTS)
        e.build_alloy_slab(slab, 0.3)
        e.set_temperature_field(models.la_front_field(box, float(slab)), "socket")
        e.refresh_rates()
        path = None
    else:
        path, d = small_deck(tmp_path, deck, (slab, 120, 120))
        tab = d.tables()
        if f2 is not None:
            tab["second_factor"] = f2
        e = Engine(box, tab, seed=29, tile=tile, tau_policy=1, events_per_pass=k)
        e.build_slab(mode, slab - slab % 24)
    e.set_schedule(schedule)
    return e, path


@pytest.mark.parametrize("case", list(CASES))
def test_agrees_with_the_colour_passes(tmp_path, case):
    out = {}
    for schedule in ("colours", "tiles", "mixed"):
        e, _ = make(tmp_path, case, "colours" if schedule == "colours" else "tiles")
        runs = [e.run(30000)]
        if schedule == "mixed":
            e.set_schedule("colours")
        runs.append(e.run(15000))
        lat, mc, bulk, void = e.store_state()
        counts, clock, lists = e.counters()
        out[schedule] = (runs, lat, mc, list(counts), clock, lists, e.diagnostics())
        print(f"[{case} {schedule}] {runs}", flush=True)
        e.close()
    want = out["colours"]
    assert want[0][0][0] >= 30000
    for schedule in ("tiles", "mixed"):
        got = out[schedule]
        assert got[0] == want[0] and got[3:] == want[3:], schedule
        assert np.array_equal(got[1], want[1]), schedule
        for k in want[2]:
            assert np.array_equal(got[2][k], want[2][k]), (schedule, k)


@pytest.mark.parametrize("case", ["SiC-f2", "CVD"])
def test_log_is_a_serial_history(tmp_path, case):
    _, _, box, _, _, _, f2 = CASES[case]
    e, path = make(tmp_path, case, "tiles")
    e.set_event_log(200000)
    n, t, stop = e.run(40000)
    log = e.event_log()
    assert len(log) == n and n >= 40000
    o = Oracle(*box)
    o.load_deck(path)
    if f2 is not None:
        o.set_second_factor(f2)
    o.apply_log(log)
    assert o.anomalies()["oob_reads"] == 0
    lat_o, mc_o, _, _ = oracle_state(o)
    lat_e, mc_e, _, _ = e.store_state(lattcoo=lat_o.copy())
    assert not np.any((lat_o != lat_e) & parity_mask(box))
    assert list_map(mc_o) == list_map(mc_e)
    o.close()
    e.close()
