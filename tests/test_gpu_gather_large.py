"""Gathers along an axis around the number of elements from which a lane has several of them."""

import numpy as np
import pytest

from raven_amd import dtype as dt
from raven_amd.nx_backend import logical

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [dt.float32, dt.uint8, dt.int64], ids=lambda d: d.name)
@pytest.mark.parametrize("rows,cols,axis", [(1, (1 << 20) - 1, 1), (1, 1 << 20, 1), (1025, 1023, 1), (1031, 1024, 0), (3, 700001, 1), (2051, 517, 1)])
def test_gather_of_a_million_elements(hip, d, rows, cols, axis):
    rng = np.random.default_rng(rows + cols)
    raw = rng.integers(0, 100, (rows, cols)).astype(d.np_storage)
    n = (rows, cols)[axis]
    ids = rng.integers(-n, n, (rows, cols)).astype(np.int32)
    t, i = hip.reshape(hip.from_host(raw, d), raw.shape), hip.reshape(hip.from_host(ids, dt.int32), ids.shape)
    assert np.array_equal(logical(hip.gather(t, i, axis)), np.take_along_axis(raw, ids % n, axis))
    turned = hip.gather(hip.permute(t, (1, 0)), hip.permute(i, (1, 0)), 1 - axis)
    assert np.array_equal(logical(turned), np.take_along_axis(raw, ids % n, axis).T)
    ids[-1, -1] = n
    with pytest.raises(RuntimeError):
        hip.gather(t, hip.reshape(hip.from_host(ids, dt.int32), ids.shape), axis)
