"""GPU: what an engine keeps between calls follows its lattice.  Many small
engines (a parameter scan) whose states and frames have been fetched hold at
most two workspaces of a fifth of their lattices' memory each on the device, and
share a few page-locked buffers on the host."""
import threading

import numpy as np
import pytest
import torch

from mulskips_amd import models
from mulskips_amd.engine import Engine

pytestmark = pytest.mark.gpu

BOX, N = (96, 96, 130), 48
LATTICE = BOX[0] // 2 * (BOX[1] // 2) * (BOX[2] + 1) * 21  # bytes


def _device_free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def _address_space():
    """This process's address space in bytes (page-locked host memory is part
    of it whether or not it counts as resident)."""
    with open("/proc/self/status") as f:
        return next(int(line.split()[1]) * 1024 for line in f if line.startswith("VmSize:"))


def _engine(seed):
    e = Engine(BOX, models.si_c1_tables(), seed=seed, tile=16)
    e.build_slab(0, 48)
    return e


def _fetch(e):
    e.frame()
    return e.store_state()


def test_many_engines_keep_little():
    first = _engine(1)  # what the process allocates once
    want = _fetch(first)
    engines = [_engine(2 + i) for i in range(N)]
    free, space = _device_free(), _address_space()
    for e in engines:
        _fetch(e)
    kept = free - _device_free()
    grown = _address_space() - space
    print(f"{N} engines of {LATTICE / 1e6:.1f} MB: kept {kept / 1e6:.1f} MB on the device, address space "
          f"+{grown / 1e6:.1f} MB", flush=True)
    # two fifths of the lattice an engine, allocations rounded up to 2 MB
    assert kept <= N * (2 * LATTICE // 5 + (2 << 20))
    # the same as device memory's addresses, and nothing an engine on the host
    assert grown <= N * (2 * LATTICE // 5 + (2 << 20)) + (128 << 20)
    # several threads at once, each with engines of its own: the buffers are not shared while in use
    out = [None] * 4

    def work(k):
        out[k] = [_fetch(engines[k]) for _ in range(8)]

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for states in out:
        for got in states:
            assert np.array_equal(got[0], want[0])
            for a, b in zip(want[1:], got[1:]):
                for key in a:
                    assert np.array_equal(a[key], b[key]), key
    for e in engines + [first]:
        e.close()
    again = _engine(5)  # the last engine gave the buffers back
    assert np.array_equal(_fetch(again)[0], want[0])
    again.close()
