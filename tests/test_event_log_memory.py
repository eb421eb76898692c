"""Engine.event_log's host memory follows the events logged, not the log's
capacity: the library's call is stood in for by one that keeps its contract
(all of the log's length, as many records as fit) on the CPU."""
import ctypes as C

import numpy as np
import pytest

from mulskips_amd import _lib
from mulskips_amd.engine import LOG_ROWS, Engine


class FakeLog:
    def __init__(self, events):
        self.log = np.zeros(events, _lib.EVENT_DTYPE)
        self.log["iter"] = np.arange(1, events + 1)

    def mskg_set_event_log(self, h, capacity):
        self.capacity = capacity
        return 0

    def mskg_get_event_log(self, h, out, cap, n):
        C.cast(n, C.POINTER(C.c_int64)).contents.value = len(self.log)
        m = min(len(self.log), cap)
        if m:
            C.memmove(out, self.log.ctypes.data, m * self.log.itemsize)
        return 0

    def mskg_destroy(self, h):
        pass


@pytest.mark.parametrize("events", [0, 1, LOG_ROWS - 1, LOG_ROWS, LOG_ROWS + 1, 3 * LOG_ROWS + 5])
def test_array_is_sized_by_the_events(events):
    e = Engine.__new__(Engine)
    e.L, e.h = FakeLog(events), None
    e.set_event_log(10 ** 10)  # 480 GB of records
    log = e.event_log()
    assert log.dtype == _lib.EVENT_DTYPE and np.array_equal(log, e.L.log)
    held = log if log.base is None else log.base
    assert len(held) <= max(events, LOG_ROWS)
