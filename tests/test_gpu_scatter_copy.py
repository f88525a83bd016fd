"""The one-pass copy and scatter of whole rows (scatter_copy) where its blocks, lists and vectors end: against a copy
followed by a scatter, bit for bit, and against a serial sum."""

import time

import numpy as np
import pytest

from helpers import same_bits
from raven_amd import dtype as dt
from raven_amd.nx_backend import logical

pytestmark = pytest.mark.gpu


def rows_of(hip, ids, cols):
    return hip.expand(hip.reshape(hip.from_host(ids.astype(np.int32), dt.int32), (len(ids), 1)), (len(ids), cols))


@pytest.mark.parametrize("d", [dt.float32, dt.bfloat16, dt.int64], ids=lambda d: d.name)
@pytest.mark.parametrize("rows,cols,n,spread", [
    (1, 8, 1, 1), (15, 1024, 60, 15), (16, 1024, 64, 2), (17, 1023, 64, 17), (600, 16, 1024, 600), (600, 16, 1025, 600),
    (600, 17, 2400, 1), (3000, 260, 2049, 3), (50257, 96, 8192, 50257), (5000, 7, 16385, 40)])
def test_equals_copy_then_scatter(hip, d, rows, cols, n, spread):
    """`spread`: how many different rows are hit; lists of up to 1024 updates and of more, in one block."""
    rng = np.random.default_rng(rows * 7 + cols + n)

    def tensor(shape):
        if d is dt.bfloat16:
            return hip.cast(hip.reshape(hip.from_host(rng.standard_normal(shape).astype(np.float32), dt.float32), shape), d)
        return hip.reshape(hip.from_host(rng.integers(-9, 9, shape).astype(d.np_storage), d), shape)

    template, updates = tensor((rows, cols)), tensor((n, cols))
    ids = rng.integers(0, spread, n) - rng.integers(0, 2, n) * rows
    index = rows_of(hip, ids, cols)
    for mode in ("add", "set"):
        got = hip.scatter(mode, False, template, index, updates, 0)
        assert hip.last_path() == "scatter_copy"
        want = hip.copy(template)
        hip._check(hip._lib.nxh_scatter(hip._h, want._desc(), index._desc(), updates._desc(), 0, {"set": 0, "add": 1}[mode]))
        same_bits(logical(got), logical(want), mode)


def test_sums_in_the_order_of_positions(hip):
    rng = np.random.default_rng(3)
    rows, cols, n = 40, 1000, 160
    t, u = rng.standard_normal((rows, cols)).astype(np.float32), rng.standard_normal((n, cols)).astype(np.float32)
    ids = rng.integers(0, 5, n)
    template = hip.reshape(hip.from_host(t, dt.float32), (rows, cols))
    got = hip.scatter("add", False, template, rows_of(hip, ids, cols), hip.reshape(hip.from_host(u, dt.float32), (n, cols)), 0)
    assert hip.last_path() == "scatter_copy"
    want = t.copy()
    for i, r in enumerate(ids):
        want[r] += u[i]
    same_bits(logical(got), want, "serial")


def two_launches(hip, mode, template, index, updates):
    out = hip.copy(template)
    hip._check(hip._lib.nxh_scatter(hip._h, out._desc(), index._desc(), updates._desc(), 0, {"set": 0, "add": 1}[mode]))
    return out


@pytest.mark.parametrize("cols", [8, 7])
@pytest.mark.parametrize("most", [15, 16, 17, 29, 1024, 1025, 3000])
def test_rows_that_many_updates_hit(hip, cols, most):
    """`most` updates of one row, next to each other and apart: those added on the way, those added after the copy, lists
    that don't take them all, and spans of positions that are halved until they do."""
    rng = np.random.default_rng(most)
    rows, n = 5000, 20000
    template = hip.reshape(hip.from_host(rng.standard_normal((rows, cols)).astype(np.float32), dt.float32), (rows, cols))
    updates = hip.reshape(hip.from_host(rng.standard_normal((n, cols)).astype(np.float32), dt.float32), (n, cols))
    for name, places in (("together", np.arange(most)), ("at the end", n - 1 - np.arange(most)), ("apart", rng.permutation(n)[:most])):
        ids = rng.integers(0, rows, n)
        ids[places] = 3
        index = rows_of(hip, ids, cols)
        for mode in ("add", "set"):
            got = hip.scatter(mode, False, template, index, updates, 0)
            assert hip.last_path() == "scatter_copy"
            same_bits(logical(got), logical(two_launches(hip, mode, template, index, updates)), f"{name} {mode}")


def seconds(hip, f):
    best = 1.0
    for _ in range(5):
        hip.synchronize()
        t = time.perf_counter()
        f()
        hip.synchronize()
        best = min(best, time.perf_counter() - t)
    return best


@pytest.mark.parametrize("mode", ["add", "set"])
@pytest.mark.parametrize("cols", [768, 770])
def test_one_row_for_all_costs_no_more_than_two_launches(hip, mode, cols):
    """As a padding token's: 8 192 updates of one row, which one block adds up (0.6 ms and 1.5, set 0.25; two launches 1.8 and
    1.9, set 0.6 and 0.9)."""
    template, updates = hip.full(dt.float32, (50257, cols), 0.0), hip.full(dt.float32, (8192, cols), 1.0)
    index = rows_of(hip, np.full(8192, 7), cols)

    one = seconds(hip, lambda: hip.scatter(mode, False, template, index, updates, 0))
    assert hip.last_path() == "scatter_copy"
    assert one < seconds(hip, lambda: two_launches(hip, mode, template, index, updates))


@pytest.mark.parametrize("rows,cols,n,one_pass", [
    (16, 16384, 16, True), (2, 16388, 2, False), (16, 32768, 16, False), (1, 262144, 4, False), (128, 65536, 128, False),
    (64, 3071, 64, True), (4, 4099, 4, False), (64, 3073, 64, False), (100, 10001, 100, False), (15, 100001, 8, False),
    (3000, 1025, 3000, True), (1000, 4099, 1000, False)])
def test_long_rows_are_not_left_to_a_few_blocks(hip, rows, cols, n, one_pass):
    """A row, or as many as are whole vectors, is one block's work at the least: past some 64 KiB it is copied by the whole chip."""
    rng = np.random.default_rng(cols)
    template = hip.reshape(hip.from_host(rng.standard_normal((rows, cols)).astype(np.float32), dt.float32), (rows, cols))
    updates = hip.reshape(hip.from_host(rng.standard_normal((n, cols)).astype(np.float32), dt.float32), (n, cols))
    index = rows_of(hip, rng.integers(0, rows, n), cols)
    for mode in ("add", "set"):
        got = hip.scatter(mode, False, template, index, updates, 0)
        assert (hip.last_path() == "scatter_copy") == one_pass, hip.last_path()
        same_bits(logical(got), logical(two_launches(hip, mode, template, index, updates)), mode)


@pytest.mark.parametrize("rows,cols,n,one_pass", [
    (1000, 2, 4000, True), (10000, 3, 40000, True), (224, 4, 896, True), (225, 7, 900, True), (120001, 4, 120000, True), (1000000, 3, 1500000, True),
    (120001, 3, 480004, True), (3300000, 2, 200000, True), (3300000, 2, 3300000, False), (8400000, 2, 8400, False)])
def test_dense_updates_of_narrow_tables(hip, rows, cols, n, one_pass):
    """Ranges that a block's list bounds, and tables whose many blocks would read more indices than the copy they save is worth."""
    rng = np.random.default_rng(n)
    template = hip.reshape(hip.from_host(rng.standard_normal((rows, cols)).astype(np.float32), dt.float32), (rows, cols))
    updates = hip.reshape(hip.from_host(rng.standard_normal((n, cols)).astype(np.float32), dt.float32), (n, cols))
    index = rows_of(hip, rng.integers(-rows, rows, n), cols)
    for mode in ("add", "set"):
        got = hip.scatter(mode, False, template, index, updates, 0)
        assert (hip.last_path() == "scatter_copy") == one_pass, hip.last_path()
        same_bits(logical(got), logical(two_launches(hip, mode, template, index, updates)), mode)


def test_dense_updates_cost_no_more_than_two_launches(hip):
    """Four updates a row of a narrow table (12 us a call among others; copied and scattered 23)."""
    rows, n = 1000, 4000
    template, updates = hip.full(dt.float32, (rows, 2), 0.0), hip.full(dt.float32, (n, 2), 1.0)
    index = rows_of(hip, np.arange(n) % rows, 2)
    one = seconds(hip, lambda: hip.scatter("add", False, template, index, updates, 0))
    assert hip.last_path() == "scatter_copy"
    assert one < seconds(hip, lambda: two_launches(hip, "add", template, index, updates))
