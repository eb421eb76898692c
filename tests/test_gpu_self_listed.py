"""GPU: sites that list themselves.  Where a neighbour's evaporation leaves a
site of coordination 1 without a reciprocal partner, its list holds the origin;
an atom deposited there takes its zig-zag candidates from the origin's record,
and with no list there (a wall) they are the site itself.  The events then visit
their own site's record among the neighbours, in list order.

Every state and event is given to the oracle too: equal lattice and lists bit
for bit, rates within the FP32 rounding of the FP64 rate (2^-24 of it, taken as
1e-7 relative), and what the oracle refuses the engine refuses.  Below a frozen
substrate's bound, an engine option that leaves the check of the coordination
out, the record is the serial rules' by hand."""
import os

import numpy as np
import pytest

from mulskips_amd import _lib
from mulskips_amd import deck as deckmod
from mulskips_amd import models
from mulskips_amd.engine import Engine, EngineError
from oracle.oracle import Oracle
from tests.helpers import list_map, oracle_state, parity_mask

pytestmark = pytest.mark.gpu

BOX = (96, 96, 96)
SITE = (63, 9, 57)  # in the vacuum above the slab, a diamond site
BONDED = (66, 12, 54)  # one of its bonds


def _tables():
    tab = models.si_c1_tables()
    tab["ptrans_zig"] = 1.0
    return tab


def _pair(tmp_path, frozen=0):
    path = os.path.join(str(tmp_path), "start.dat")
    # the deck gives the tables; its own shape has no atoms (extents below zero)
    deckmod.write_start_dat(deckmod.deck_from_tables(_tables(), "C", [-20, -20, -20], idum=7), path)
    o = Oracle(*BOX)
    o.load_deck(path)
    e = Engine(BOX, _tables(), seed=3, tile=24, frozen_below_z=frozen)
    e.build_slab(0, 24)
    return o, e


def _add(state, sites):
    """The state with more sites: (position, LattCoo word, neighbour list, event)."""
    lat, mc, bulk, void = state
    lat = lat.copy()
    for (x, y, z), word, _, _ in sites:
        lat[z, y, x] = word
    mc = {"xyz": np.concatenate([mc["xyz"], [s[0] for s in sites]]).astype(np.int32),
          "nn": np.concatenate([mc["nn"].reshape(-1, 4, 3), [s[2] for s in sites]]).astype(np.int32),
          "event": np.concatenate([mc["event"], [s[3] for s in sites]]).astype(np.int32),
          "prob": np.concatenate([np.maximum(mc["prob"], 1e-3), [1e-3] * len(sites)])}  # frozen atoms: none
    return lat, mc, bulk, void


def _event(site, itrans, coor, arm=-1):
    log = np.zeros(1, _lib.EVENT_DTYPE)
    log["iter"], log["site"], log["itrans"], log["arm"] = 1, site, itrans, arm
    log["coor"], log["rtot"], log["time"] = coor, 1.0, 1.0
    return log


def _word(species, coor):
    return ((1 << 23) | (species << 27) if species else 0) | (coor << 24)


UNFIXED = [(0, 0, 0)] * 4


def test_deposition_that_lists_itself_is_refused(tmp_path):
    o, e = _pair(tmp_path)
    state = _add(e.store_state(), [(SITE, _word(0, 1), UNFIXED, 1)])
    o.load_state(*state)
    e.load_state(*state)
    log = _event(SITE, 1, 1, arm=0)
    with pytest.raises(RuntimeError, match="Get Prob Error"):
        o.apply_log(log)
    with pytest.raises(EngineError, match="coordination inconsistent"):
        e.replay(log)
    o.close()
    e.close()


def test_deposition_below_the_frozen_bound(tmp_path):
    """Serial rules: the site takes the species at coordination 1; the wall at
    the origin adds one; each of the three visits of the site itself adds one to
    its record's coordination (below 4) and one to the count: 1 + 1 + 3."""
    o, e = _pair(tmp_path, frozen=SITE[2] + 1)
    state = _add(e.store_state(), [(SITE, _word(0, 1), UNFIXED, 1)])
    e.load_state(*state)
    e.replay(_event(SITE, 1, 1, arm=0))
    lat, mc, bulk, _ = e.store_state()
    x, y, z = SITE
    assert lat[z, y, x] == _word(1, 5)
    assert tuple(SITE) in list_map(bulk) and tuple(SITE) not in list_map(mc)
    assert list_map(bulk)[SITE] == (0, 0, 0) + 3 * SITE
    o.close()
    e.close()


# the self-listing atom's list (coordination 2 with its bonded atom, at the entry given)
LISTS = {
    "bonded first": [BONDED, SITE, (0, 0, 0), (0, 0, 0)],
    "itself first": [SITE, BONDED, (0, 0, 0), (0, 0, 0)],
    "twice itself": [BONDED, SITE, SITE, (0, 0, 0)],
}


@pytest.mark.parametrize("name", list(LISTS))
def test_evaporation_of_a_self_listing_atom(tmp_path, name):
    o, e = _pair(tmp_path)
    nn = LISTS[name]
    coor = 1 + sum(n == SITE for n in nn)
    other = [SITE, (69, 15, 57), (69, 9, 51), (63, 15, 51)]
    # the walls at the origin count for a listed origin: leave it empty in both
    state = list(e.store_state())
    state[0] = state[0].copy()
    state[0][0, 0, 0] = 0
    state = _add(state, [(SITE, _word(1, coor), nn, 4), (BONDED, _word(1, 1), other, 4)])
    o.load_state(*state)
    o.refresh_all()
    e.load_state(*state)
    e.refresh_rates()
    log = _event(SITE, 4, coor)
    try:
        o.apply_log(log)
    except RuntimeError as err:
        with pytest.raises(EngineError):
            e.replay(log)
        print(f"[{name}] both refuse: {err}")
    else:
        e.replay(log)
        lat_o, mc_o, bulk_o, void_o = oracle_state(o)
        lat_e, mc_e, bulk_e, void_e = e.store_state(lattcoo=lat_o.copy())
        assert np.count_nonzero((lat_o != lat_e) & parity_mask(BOX)) == 0
        for a, b in ((mc_o, mc_e), (bulk_o, bulk_e), (void_o, void_e)):
            assert list_map(a) == list_map(b)
        cls, rate = e.site_rates(mc_o["xyz"])
        keep = cls != 6
        np.testing.assert_allclose(rate[keep], mc_o["prob"][keep], rtol=1e-7)
    o.close()
    e.close()
