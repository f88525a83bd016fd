"""A factorisation or a solve answers for its own matrices only, whatever the calls before it found and however many
matrices it has: calls that fail and calls that succeed in turn, nothing waited for in between."""

import numpy as np
import pytest

from helpers import same_bits
from raven_amd import dtype as dt
from raven_amd.nx_backend import logical

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [dt.float32, dt.complex128], ids=lambda d: d.name)
@pytest.mark.parametrize("batch,n,nrhs", [(1, 1, 1), (1, 16, 3), (1, 17, 40), (3, 33, 5), (1, 515, 17), (2, 130, 2), (1, 1100, 2)])
def test_failures_stay_with_their_calls(hip, d, batch, n, nrhs):
    rng = np.random.default_rng(n)

    def tensor(x):
        return hip.reshape(hip.from_host(x.astype(d.np_storage), d), x.shape)

    low = np.tril(rng.uniform(-1, 1, (batch, n, n)) / n) + 2 * np.eye(n)
    good, b = tensor(low @ low.transpose(0, 2, 1)), tensor(rng.uniform(-1, 1, (batch, n, nrhs)))
    bad = np.array(low)
    bad[-1, n - 1, n - 1] = 0
    triangle, singular = tensor(low), tensor(bad)
    bad = low @ low.transpose(0, 2, 1)
    bad[0, n // 2, n // 2] = -1
    indefinite = tensor(bad)

    def solve(a, unit=False):
        return hip.triangular_solve(a, b, upper=False, transpose=False, unit_diag=unit)

    first = logical(hip.cholesky(good)), logical(solve(triangle)), logical(solve(singular, True))
    for _ in range(2):
        with pytest.raises(RuntimeError, match="not positive definite"):
            hip.cholesky(indefinite)
        factor = hip.cholesky(good)
        with pytest.raises(RuntimeError, match="singular"):
            solve(singular)
        x = solve(triangle)
        with pytest.raises(RuntimeError, match="singular"):
            solve(singular)
        unit = solve(singular, True)  # its diagonal is not read
        for got, want in zip((factor, x, unit), first):
            same_bits(logical(got), want, "the same call before")
    assert np.allclose(np.matmul(low, first[1]), logical(b), atol=1e-3 * n)
