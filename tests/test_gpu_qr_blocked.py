"""QR by panels: at the edges of its panels, waves and register forms."""

import numpy as np
import pytest

from helpers import logical
from raven_amd import dtype as dt

pytestmark = pytest.mark.gpu
EPS = {dt.float64: 2.0**-53, dt.float32: 2.0**-24}


@pytest.mark.parametrize("d", [dt.float64, dt.float32], ids=lambda d: d.name)
@pytest.mark.parametrize("m,n", [(1, 1), (1, 7), (2, 1), (5, 5), (15, 16), (16, 16), (17, 17), (33, 31), (64, 64), (65, 65), (80, 20),
                                 (20, 80), (129, 128), (256, 30), (257, 48), (513, 17), (1024, 40), (1025, 33), (2048, 16), (2049, 3),
                                 (300, 300)])
def test_factors(hip, d, m, n):
    rng = np.random.default_rng(m * 3 + n)
    a = rng.standard_normal((2, m, n)).astype(d.np_storage)
    x = hip.reshape(hip.from_host(a, d), a.shape)
    k = min(m, n)
    for reduced in (True, False):
        q, r = (logical(t).astype(np.float64) for t in hip.qr(x, reduced))
        assert hip.last_path() == ("qr_blocked" if m <= 2048 else "qr_householder_wide")
        assert q.shape == (2, m, k if reduced else m) and r.shape == (2, k if reduced else m, n)
        assert np.all(np.tril(r, -1) == 0)
        # k reflectors of m rows, each a rounding or two of every element it meets; the factors are stored in d
        bound = 8 * EPS[dt.float64] * (k + 8) + 4 * EPS[d]
        assert np.max(np.abs(q.swapaxes(1, 2) @ q - np.eye(q.shape[2]))) <= bound * np.sqrt(m)
        assert np.max(np.linalg.norm(q @ r - a, axis=(1, 2)) / np.linalg.norm(a, axis=(1, 2))) <= bound
        want = np.linalg.qr(a.astype(np.float64), "reduced")[1]  # the reflectors' own signs
        assert np.all(np.sign(np.diagonal(r, axis1=1, axis2=2)) == np.sign(np.diagonal(want, axis1=1, axis2=2)))
    t = hip.permute(hip.reshape(hip.from_host(np.ascontiguousarray(a.swapaxes(1, 2)), d), (2, n, m)), (0, 2, 1))
    assert np.array_equal(logical(hip.qr(t)[1]).astype(np.float64), r[:, :k])


def test_columns_without_a_reflector(hip):
    """A column that is zero below the diagonal takes none: a triangular input comes back as it is."""
    for n in (7, 40, 100):
        a = np.triu(np.random.default_rng(n).standard_normal((n, n)))
        a[:, 3] = 0.0
        q, r = hip.qr(hip.reshape(hip.from_host(a, dt.float64), a.shape))
        assert np.array_equal(logical(q), np.eye(n)) and np.array_equal(logical(r), a)
    a = np.zeros((70, 20))
    q, r = hip.qr(hip.reshape(hip.from_host(a, dt.float64), a.shape))
    assert np.array_equal(logical(q), np.eye(70)[:, :20]) and np.array_equal(logical(r), a[:20])


def test_many_matrices(hip):
    rng = np.random.default_rng(1)
    a = rng.standard_normal((3000, 20, 18))
    q, r = (logical(t) for t in hip.qr(hip.reshape(hip.from_host(a, dt.float64), a.shape)))
    assert np.max(np.abs(q @ r - a)) < 1e-13 and np.max(np.abs(q.swapaxes(1, 2) @ q - np.eye(18))) < 1e-13
