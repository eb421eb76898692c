"""GPU: the wave-cooperative event execution at the places where its lanes
play different roles, against the oracle's serial update rules.

* a frozen substrate, whose own sites fill without a rate: the site's record
  and a neighbour's first list entry are stored by lanes of one quad;
* the second-neighbour term, whose shell shares the quads' rate evaluation;
* coverage species: a covered site of coordination 1 lists the origin three
  times, so its neighbours are visited in order, a round each;
* coverage species with the second-neighbour term: the shell in a round of
  its own.

The engine's run is logged; the oracle applies the log, and a second engine
replays it.  Lattice, list membership and neighbour lists are equal bit for
bit, rates within the FP32 rounding of the FP64 rate (2^-24 of it, taken as
1e-7 relative).  With coverage species and the second-neighbour term
together, an option the reference lacks, engine and oracle refresh an atom
beside a covered site at different events, so there the rates of the run and
of the replay are compared with each other instead.
"""
import numpy as np
import pytest

from mulskips_amd.engine import Engine
from oracle.oracle import Oracle
from tests.helpers import list_map, oracle_state, parity_mask, small_deck

pytestmark = pytest.mark.gpu

F2 = np.exp(-np.arange(13) * 0.05 / (8.617333262e-5 * 1600.0))
# name: (deck, slab builder mode, box, lens, frozen below z, second-neighbour factors, tile)
CASES = {
    "Si-frozen": ("Si-SL", 0, (96, 96, 144), (72, 120, 120), 73, None, 16),
    "SiC-f2-frozen": ("surface", 1, (96, 96, 288), (72, 72, 72), 73, F2, 24),
    "CVD": ("CVD-Si-SiH2", 0, (96, 96, 192), (72, 120, 120), 0, None, 24),
    "CVD-f2-frozen": ("CVD-Si-SiH2", 0, (96, 96, 192), (72, 120, 120), 60, F2, 24),
}


@pytest.mark.parametrize("case", list(CASES))
def test_run_and_replay_follow_the_serial_rules(tmp_path, case):
    deck, mode, box, lens, frozen, f2, tile = CASES[case]
    path, d = small_deck(tmp_path, deck, lens)
    o = Oracle(*box)
    o.load_deck(path)
    if frozen:
        o.set_frozen(frozen)
    tab = d.tables()
    if f2 is not None:
        o.set_second_factor(f2)
        tab["second_factor"] = f2

    def make():
        e = Engine(box, tab, seed=7, tile=tile, events_per_pass=4.0, tau_policy=1, frozen_below_z=frozen)
        e.build_slab(mode, lens[0] - lens[0] % 24)
        return e

    eng = make()
    eng.set_event_log(100000)
    n, t, stop = eng.run(30000)
    log = eng.event_log()
    assert len(log) == n and n > 1000 and stop in (0, 1)
    again = make()
    again.replay(log)
    o.apply_log(log)
    assert o.anomalies()["oob_reads"] == 0
    lat_o, mc_o, bulk_o, void_o = oracle_state(o)
    m = parity_mask(box)
    rates = []
    for e in (eng, again):
        lat_e, mc_e, bulk_e, void_e = e.store_state(lattcoo=lat_o.copy())
        assert np.count_nonzero((lat_o != lat_e) & m) == 0
        for a, b in ((mc_o, mc_e), (bulk_o, bulk_e), (void_o, void_e)):
            ma, mb = list_map(a), list_map(b)
            assert ma.keys() == mb.keys() and all(ma[k] == mb[k] for k in ma)
        cls, rate = e.site_rates(mc_o["xyz"])
        # isolated atoms' rates follow the run's own total; frozen atoms have none
        keep = (cls != 6) & ((mc_o["xyz"][:, 2] >= frozen) | (cls != 0))
        assert keep.sum() > 100
        if case == "CVD-f2-frozen":
            rates.append(rate[keep])
        else:
            np.testing.assert_allclose(rate[keep], mc_o["prob"][keep], rtol=1e-7)
        e.close()
    if rates:
        np.testing.assert_array_equal(rates[0], rates[1])
    o.close()
