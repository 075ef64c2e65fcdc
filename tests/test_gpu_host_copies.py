"""Host arrays to and from the device: every value arrives, whatever the size.

Large arrays take a path of their own (pinned chunks moved by several threads;
one copy at a time, the others as plain copies), grids with open directions
that are no multiple of 8 are padded on the way: shapes below and above the
path's limits, padded and not, and from several threads at once.  Copies are
compared bit for bit.
"""
import threading

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

SHAPES = [(16, 16, 16), (64, 64, 56), (96, 96, 104), (97, 89, 111), (9, 17, 33), (61, 66, 71)]


def _state(shape, seed):
    return np.asfortranarray(np.random.default_rng(seed).standard_normal(shape + (5,)))


def _scheme(shape):
    return tuple(O.OPEN if n % 8 else O.PERIODIC for n in shape)


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("precision", [0, 1])  # FP64, FP32-mixed
def test_state_round_trip(shape, precision):
    from public_amd import Cruna
    with Cruna(shape, (0.1,) * 3, scheme=_scheme(shape), precision=precision) as g:
        for seed in (1, 2):
            q = _state(shape, seed)
            g.set_state(q)
            assert np.array_equal(g.get_state(), q)
            q[...] = 0.0  # the array is the caller's again once set_state returns
            assert np.array_equal(g.get_state(), _state(shape, seed))


def test_state_round_trips_from_threads():
    from public_amd import Cruna
    shape = (96, 96, 104)
    got = {}

    def one(k):
        with Cruna(shape, (0.1,) * 3) as g:
            g.set_state(_state(shape, k))
            got[k] = g.get_state()

    ts = [threading.Thread(target=one, args=(k,)) for k in range(3)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for k in range(3):
        assert np.array_equal(got[k], _state(shape, k))
