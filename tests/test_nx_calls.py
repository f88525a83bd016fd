"""The host path in C (raven_amd/host_c/nx_calls.c): every form of argument the calls take, their errors,
the storage they give back; and the views that remember their movements."""

import gc
import threading
import weakref

import numpy as np
import pytest

from raven_amd import dtype as dt
from raven_amd.nx_backend import logical
from raven_amd.view import View


def test_remembered_movements_are_the_movements():
    for shape in ((), (1,), (3, 1), (2, 3, 4), (0, 2), (1, 5, 1)):
        v = View.create(shape)
        for _ in range(3):  # made, remembered, found
            for name, args in (("permute", [tuple(range(len(shape)))[::-1]]), ("expand", [shape, (7,) * len(shape)]),
                               ("reshape", [shape, (int(np.prod(shape)),), list(shape)[::-1], (-1, 5), (999,)])):
                for arg in args:
                    try:
                        want = getattr(View, "_" + name)(v, arg)
                    except ValueError as e:
                        with pytest.raises(ValueError, match="^" + name):
                            getattr(v, name)(arg)
                        assert str(e).startswith(name)
                        continue
                    got = getattr(v, name)(arg)
                    assert got == want and got.offset == want.offset, (shape, name, arg)
    v = View.create((1, 6))
    for n in range(1, 100):
        assert v.expand((n, 6)).strides == (0 if n > 1 else 6, 1)
    assert len(v.derived) <= 16
    assert View((2, 3), (3, 1), 0).expand((2, 3)) == View.create((2, 3))


@pytest.mark.gpu
def test_forms_of_arguments(hip):
    x = hip.reshape(hip.from_host(np.arange(24, dtype=np.float32), dt.float32), (2, 3, 4))
    n = np.arange(24, dtype=np.float32).reshape(2, 3, 4)
    for axes in ([0], (2,), [0, 2], [2, 0], np.array([1]), [np.int64(1)], (0, 1, 2), [], range(2)):
        want = n.sum(tuple(int(a) for a in axes))
        assert np.array_equal(logical(hip.reduce("sum", axes, x)), want) and hip.reduce("sum", axes, x).shape == want.shape
    assert np.array_equal(logical(hip.binary(op="add", x=x, y=x)), n + n)
    assert np.array_equal(logical(hip.cast(x, dtype=dt.int32)), n.astype(np.int32))
    assert np.array_equal(logical(hip.where(hip.compare("cmplt", x, x), x, if_false=x)), n)
    for value in (2, 2.0, np.float64(2), np.array([2], np.float32), np.array(2, np.float32)):
        for shape in ((2, 3), [2, 3], (np.int64(2), 3)):
            f = hip.full(dt.float32, shape, value)
            assert f.shape == (2, 3) and np.all(logical(f) == 2)
    assert logical(hip.full(dt.float32, (), 3.0)) == 3
    y = hip.permute(x, (0, 2, 1))
    assert np.array_equal(logical(hip.matmul(x, y)), n @ n.swapaxes(1, 2))
    w = hip.reshape(hip.from_host(np.ones(4, np.float32), dt.float32), (4, 1))
    assert np.array_equal(logical(hip.matmul(x=x, y=w)), n @ np.ones((4, 1), np.float32))  # a batch that broadcasts

    class Foreign:  # anything that describes itself is an operand
        shape, dtype = x.shape, x.dtype

        def _desc(self):
            return x._desc()

    assert np.array_equal(logical(hip.unary("neg", Foreign())), -n)
    assert np.array_equal(logical(hip.binary("mul", x, Foreign())), n * n)
    assert repr(x) == "Tensor(float32, shape=(2, 3, 4), strides=(12, 4, 1), offset=0)"
    assert x._desc() is x._desc() and x._desc().data == x.buffer.ptr


@pytest.mark.gpu
def test_errors(hip):
    x = hip.full(dt.float32, (2, 3), 1.0)
    empty = hip.buffer(dt.float32, (2, 0))
    for call, kind in ((lambda: hip.binary("nope", x, x), ValueError), (lambda: hip.binary("add", x), TypeError),
                       (lambda: hip.unary("neg", x=x, y=x), TypeError), (lambda: hip.unary("neg", z=x), TypeError),
                       (lambda: hip.unary("neg", 3), AttributeError), (lambda: hip.reduce("max", [1], empty), ValueError),
                       (lambda: hip.reduce("sum", [5], x), (ValueError, IndexError)), (lambda: hip.matmul(x, x), ValueError),
                       (lambda: hip.full(dt.float32, (2,), np.zeros(2, np.float32)), ValueError),
                       (lambda: hip.binary("add", x, hip.full(dt.float32, (3, 2), 1.0)), ValueError)):
        before = hip.memory_stats()["in_use"]
        with pytest.raises(kind):
            call()
        assert hip.memory_stats()["in_use"] == before
    assert np.all(logical(hip.reduce("sum", [1], empty)) == 0)


@pytest.mark.gpu
def test_storage_goes_back_and_threads(hip):
    gc.collect()  # what an earlier test's exceptions still hold
    before = hip.memory_stats()["in_use"]
    t = hip.full(dt.float32, (1000,), 1.0)
    gone = []
    ref = weakref.ref(t.buffer, gone.append)
    view = hip.reshape(t, (10, 100))
    del t
    assert ref() is view.buffer and hip.memory_stats()["in_use"] > before
    del view
    assert gone and hip.memory_stats()["in_use"] == before
    wrong = []

    def work(k):
        a = hip.full(dt.float32, (64, 64), float(k))
        for _ in range(200):
            s = hip.reduce("sum", [1], hip.binary("add", a, a))
        if not np.all(logical(s) == 128 * k):
            wrong.append(k)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not wrong and hip.memory_stats()["in_use"] == before
