"""An index out of range is reported by the gather that met it, whatever part of the launch looks through the indices."""

import threading

import numpy as np
import pytest

from helpers import same_bits
from raven_amd import dtype as dt
from raven_amd.nx_backend import logical

pytestmark = pytest.mark.gpu


def rows_of(hip, ids, cols):
    return hip.expand(hip.reshape(hip.from_host(ids.astype(np.int32), dt.int32), (len(ids), 1)), (len(ids), cols))


@pytest.mark.parametrize("n", [1, 255, 16384, 16385, 40000])
def test_gather_reports_an_index_at_either_end(hip, n):
    """Up to 16 384 indices are looked through by one block, more by those that move the rows."""
    table = hip.full(dt.float32, (100, 4), 3.0)
    good = np.zeros(n, np.int64)
    for at in (0, n - 1):
        for bad in (100, -101):
            ids = good.copy()
            ids[at] = bad
            with pytest.raises(RuntimeError):
                hip.gather(table, rows_of(hip, ids, 4), 0)
            same_bits(logical(hip.gather(table, rows_of(hip, good - 100 * (n > 1), 4), 0)), np.full((n, 4), 3.0, np.float32), "the next call")


def test_a_sorted_scatter_answers_for_its_own_indices(hip):
    """It lets other calls of the context in between its steps: gathers that fail there, from another thread, neither hide
    its own index out of range nor lend it theirs."""
    n = 1 << 16
    zeros, ones, table = hip.full(dt.float32, (5000,), 0.0), hip.full(dt.float32, (n,), 1.0), hip.full(dt.float32, (100, 4), 3.0)
    ids = np.arange(n, dtype=np.int32) % 5000
    good = hip.from_host(ids, dt.int32)
    ids[n // 2] = 5000
    bad = hip.from_host(ids, dt.int32)
    wrong = rows_of(hip, np.full(16385, 100), 4)
    answers, stop = [], threading.Event()

    def gathers():
        while not stop.is_set():
            try:
                hip.gather(table, wrong, 0)
                answers.append("a gather found its indices in range")
            except RuntimeError:
                pass

    t = threading.Thread(target=gathers)
    t.start()
    try:
        for _ in range(200):
            with pytest.raises(RuntimeError):
                hip.scatter("add", False, zeros, bad, ones, 0)
            hip.scatter("add", False, zeros, good, ones, 0)
            assert hip.last_path() == "scatter_sorted"
    finally:
        stop.set()
        t.join()
    assert not answers
