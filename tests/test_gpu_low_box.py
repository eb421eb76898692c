"""GPU: SiC with the second-neighbour term in boxes lower and barely higher
than two shell steps (LenZ 10..14), where the shell of a surface atom reaches
past the top plane.  The oracle runs the serial loop from the engine's slab;
the engine replays its log: lattice and lists are equal bit for bit, rates
within the FP32 rounding of the FP64 rate (2^-24 of it, taken as 1e-7
relative).  The engine's own run from the same slab ends without an error."""
import os

import numpy as np
import pytest

from mulskips_amd import deck as deckmod
from mulskips_amd import models
from mulskips_amd.engine import Engine
from oracle.oracle import Oracle
from tests.helpers import list_map, oracle_state, parity_mask

pytestmark = pytest.mark.gpu

F2 = np.exp(-np.arange(13) * 0.05 / (8.617333262e-5 * 1600.0))
SLAB, FROZEN = 9, 6


@pytest.mark.parametrize("lz", [10, 11, 12, 14])
def test_replay_follows_the_oracle(tmp_path, lz):
    box = (96, 96, lz)
    tab = models.sic_c2_tables(temperature=1600.0)
    path = os.path.join(str(tmp_path), "start.dat")
    # the deck gives the tables; its own shape has no atoms (extents below zero)
    deckmod.write_start_dat(deckmod.deck_from_tables(tab, "C", [-20, -20, -20], idum=7), path)
    tab["second_factor"] = F2
    e = Engine(box, tab, seed=7, tile=24, tau_policy=1, events_per_pass=2.0, frozen_below_z=FROZEN)
    e.build_slab(1, SLAB)
    o = Oracle(*box)
    o.load_deck(path)
    o.set_frozen(FROZEN)
    o.set_second_factor(F2)
    o.load_state(*e.store_state())
    o.refresh_all()
    log = o.step(5000)
    assert len(log) == 5000
    e.replay(log)
    lat_o, mc_o, bulk_o, void_o = oracle_state(o)
    lat_e, mc_e, bulk_e, void_e = e.store_state(lattcoo=lat_o.copy())
    assert np.count_nonzero((lat_o != lat_e) & parity_mask(box)) == 0
    for a, b in ((mc_o, mc_e), (bulk_o, bulk_e), (void_o, void_e)):
        ma, mb = list_map(a), list_map(b)
        assert ma.keys() == mb.keys() and all(ma[k] == mb[k] for k in ma)
    cls, rate = e.site_rates(mc_o["xyz"])
    keep = (cls != 6) & (cls != 0)  # isolated atoms' rates follow the run's own total; frozen atoms have none
    assert keep.sum() > 100 and np.all(mc_o["xyz"][cls == 0][:, 2] < FROZEN)
    np.testing.assert_allclose(rate[keep], mc_o["prob"][keep], rtol=1e-7)
    o.close()
    e.build_slab(1, SLAB)
    n, t, stop = e.run(5000)
    assert n >= 5000 and t > 0.0 and stop == 0
    e.close()
