"""An index out of range is reported by the gather that met it, whatever part of the launch looks through the indices."""

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
