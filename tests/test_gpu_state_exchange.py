"""GPU: LattCoo and the particle lists in and out.  A stored state loads back
to the same state where it takes one piece and where it takes several; a list
that names a site twice gives it its last record; what cannot be loaded leaves
the engine as it was."""
import numpy as np
import pytest

from mulskips_amd import models
from mulskips_amd.engine import Engine, EngineError

pytestmark = pytest.mark.gpu


def _same(a, b):
    assert np.array_equal(a[0], b[0])
    for x, y in zip(a[1:], b[1:]):
        for k in x:
            assert np.array_equal(x[k], y[k]), k


def _lists_by_host(lat):
    """Atoms and vacancies counted from LattCoo's words."""
    occ, cov, coor = (lat >> 23) & 1, lat & 255, (lat >> 24) & 7
    atom = (occ == 1) & (cov == 0)
    n_mc_atoms = np.count_nonzero((atom & (coor <= 3)))
    return n_mc_atoms, np.count_nonzero(atom & (coor > 3)), np.count_nonzero((lat >= 0) & (occ == 0) & (coor == 4))


# the store's pieces hold 2^24 points: one, two (the second short); the load
# takes LattCoo whole up to 2 GiB, else in pieces
@pytest.mark.parametrize("box,tile", [((96, 96, 131), 16), ((480, 480, 299), 24), ((1536, 1440, 250), 24)])
def test_round_trip(box, tile):
    a = Engine(box, models.si_c1_tables(), seed=5, tile=tile, tau_policy=1, events_per_pass=4.0)
    b = Engine(box, models.si_c1_tables(), seed=5, tile=tile)
    a.build_slab(0, 48)
    a.run(box[0] * box[1] // 16)
    state = a.store_state()
    lat, mc, bulk, void = state
    n_mc_atoms, n_bulk, n_void = _lists_by_host(lat)
    x, y, z = mc["xyz"].T
    word = lat[z, y, x]
    assert np.count_nonzero(((word >> 23) & 1) == 1) == n_mc_atoms
    assert len(bulk["xyz"]) == n_bulk and len(void["xyz"]) == n_void
    g = (mc["xyz"][:, 2].astype(np.int64) * box[1] + mc["xyz"][:, 1]) * box[0] + mc["xyz"][:, 0]
    assert np.all(np.diff(g) > 0)
    b.load_state(*state)
    _same(state, b.store_state())
    # words that are there already, and others, are both right in the end
    full = np.full((a.stored_planes, box[1], box[0]), 7, np.int32)
    out = b.store_state(lattcoo=full)[0]
    i = np.arange(box[0]) & 1
    for zz in (0, 3, 46, 47, 48, box[2]):
        for yy in (0, 1, box[1] - 1):
            on = (i == (zz & 1)) & ((yy & 1) == (zz & 1))
            assert np.array_equal(out[zz, yy][on], lat[zz, yy][on]) and np.all(out[zz, yy][~on] == 7)
    a.close()
    b.close()


def test_a_site_listed_twice():
    box = (96, 96, 130)
    a, b, c = (Engine(box, models.si_c1_tables(), seed=5) for _ in range(3))
    a.build_slab(0, 48)
    lat, mc, bulk, void = a.store_state()
    twice = {k: np.concatenate([v[3:6], v]) for k, v in mc.items()}  # the first three are named again later
    twice["prob"][:3] = 77.0
    twice["nn"][:3] = mc["nn"][:1] * 0
    b.load_state(lat, twice, bulk, void)
    c.load_state(lat, mc, bulk, void)
    _same(b.store_state(), c.store_state())
    both = {k: np.concatenate([v, mc[k][:2]]) for k, v in bulk.items()}  # MC particles named as bulk, too
    both["nn"][-2:] = 0
    b.load_state(lat, mc, both, void)
    out = b.store_state()[1]
    assert np.all(out["nn"][:2] == 0) and np.array_equal(out["nn"][2:], mc["nn"][2:])
    assert np.array_equal(out["prob"], mc["prob"])
    for e in (a, b, c):
        e.close()


def test_refused_states_change_nothing():
    box = (96, 96, 130)
    e = Engine(box, models.si_c1_tables(), seed=5)
    e.build_slab(0, 48)
    state = e.store_state()
    lat, mc, bulk, void = state
    bad = lat.copy()
    bad[60, 2, 4] = 5  # no such coverage species
    bad[90, 0, 0] = 1 << 27
    with pytest.raises(EngineError, match=r"LattCoo\(4,2,60\)"):
        e.load_state(bad, mc, bulk, void)
    off = {k: v.copy() for k, v in bulk.items()}
    off["xyz"][4] = (1, 2, 3)
    with pytest.raises(EngineError, match="list 1 record 4"):
        e.load_state(lat, mc, off, void)
    zero = {k: v.copy() for k, v in mc.items()}
    zero["prob"][9] = 0.0
    with pytest.raises(EngineError, match="record 9 has a non-positive rate"):
        e.load_state(lat, zero, bulk, void)
    _same(state, e.store_state())
    with pytest.raises(EngineError, match="capacity too small"):
        e.store_state(capacity=(len(mc["xyz"]) - 1, len(bulk["xyz"]), 0))
    e.close()
