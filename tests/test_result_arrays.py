"""Which arrays of the caller a solver writes in place, and that the others
take or refuse the result as an assignment does; arguments refused before the
library is called."""
import ctypes
import types

import numpy as np
import pytest

import iroiro_amd as ii
from iroiro_amd import _lib


def deliver(a, x):
    """What the solver classes do with a result x for the caller's array a."""
    y = _lib.result_f64(a, x.size)
    ctypes.memmove(y.ctypes.data, x.ctypes.data, x.nbytes)  # the library's write
    if y is not a:
        a[...] = y


def test_plain_arrays_in_place():
    a = np.zeros(6)
    assert _lib.result_f64(a, 6) is a
    deliver(a, np.arange(6.0))
    assert np.array_equal(a, np.arange(6.0))


@pytest.mark.parametrize("a", [np.zeros(6, np.float32), np.zeros(12)[::2], np.zeros((1, 6)),
                               np.zeros(6, ">f8"), np.zeros((6, 1)).T,
                               np.frombuffer(bytearray(49), np.float64, 6, 1)])
def test_other_arrays_by_assignment(a):
    assert _lib.result_f64(a, 6) is not a
    deliver(a, np.arange(6.0))
    assert np.array_equal(np.ravel(a), np.arange(6.0))


def test_masked_arrays_take_the_values_as_an_assignment():
    a = np.ma.array(np.zeros(6), mask=[True] * 6)
    deliver(a, np.arange(6.0))
    assert not a.mask.any() and np.array_equal(a.data, np.arange(6.0))


@pytest.mark.parametrize("shape", [(2, 3), (6, 1), (3, 2, 1), (5,)])
def test_shapes_that_an_assignment_refuses(shape):
    a = np.zeros(shape)
    with pytest.raises(ValueError):
        deliver(a, np.arange(6.0))
    assert not a.any()


@pytest.mark.parametrize("bs,ys", [([], []), ([np.zeros(192)], []),
                                   ([np.zeros(192)], [np.zeros(180)])])
def test_loss_grad_refuses_pairs_that_do_not_match(bs, ys):
    """Before anything reaches the device: no pairs, pairs of different number
    or size are a ValueError."""
    ctx = types.SimpleNamespace(V=16, handle=None)
    with pytest.raises(ValueError):
        ii.LearnedPreconditioner(ctx).loss_grad(bs, ys)


def test_loss_grad_is_one_call_of_the_library():
    """Several pairs, in arrays of their own: one call, that is one download and
    one synchronisation, and no copy that joins them."""
    calls = []

    def record(handle, n, bs, ys, loss, grads):
        calls.append([[ctypes.addressof(v[k].contents) for k in range(n)] for v in (bs, ys)])
        return _lib.II_OK

    ctx = types.SimpleNamespace(V=16, handle=None, check=lambda st, what: None)
    net = ii.LearnedPreconditioner(ctx)
    net._L = lambda: types.SimpleNamespace(ii_net_loss_grad_pairs=record)
    bs, ys = list(np.zeros((3, 192))), [np.zeros(192) for _ in range(3)]
    net.loss_grad(bs, ys)
    assert calls == [[[v.ctypes.data for v in bs], [v.ctypes.data for v in ys]]]
