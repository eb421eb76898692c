"""GPU: walls are neither MC particles nor vacancies in the particle lists,
whatever coordination the host's LattCoo gives their words."""
import numpy as np
import pytest

from mulskips_amd import models
from mulskips_amd.engine import Engine

pytestmark = pytest.mark.gpu


def test_walls_of_any_coordination_stay_out_of_the_lists():
    box = (96, 96, 130)
    a, b = (Engine(box, models.si_c1_tables(), seed=5, tile=16) for _ in range(2))
    a.build_slab(0, 48)
    a.run(2000)
    lat, mc, bulk, void = a.store_state()
    marked = lat.copy()
    z = np.arange(box[2] + 1)[:, None, None]
    coor = np.broadcast_to(z % 5, lat.shape).astype(np.int32)  # 0..4, plane by plane
    wall = (lat & 255) == 113
    marked[wall] |= coor[wall] << 24
    assert np.count_nonzero(((marked >> 24) & 7 == 4) & wall) > 0
    b.load_state(marked, mc, bulk, void)
    out = b.store_state(lattcoo=marked.copy())
    assert np.array_equal(out[0], marked)
    for want, got in zip((mc, bulk, void), out[1:]):
        for k in want:
            assert np.array_equal(want[k], got[k]), k
    a.close()
    b.close()
