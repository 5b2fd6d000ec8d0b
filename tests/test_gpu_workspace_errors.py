"""The context's workspace under threads, calls that fail among them."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from pycd_amd import _native
from tests.test_gpu_workspace import CELL, _lists, _table

pytestmark = pytest.mark.gpu


def _too_full(n):
    """A list whose shells hold more than the room given, which the call
    refuses after its kernel has run."""
    pos = np.random.default_rng(n).uniform(size=(n, 3)) @ (20 * CELL)
    idx = np.arange(n, dtype=np.int64)
    count = np.empty((n, 1), dtype=np.int32)
    index = np.empty((n, 1, 1), dtype=np.int32)
    vec = np.empty((n, 1, 1, 3))
    lo, hi = np.array([-1.0]), np.array([40.0])
    cell = np.ascontiguousarray(20 * CELL)
    pbc = np.ones(3, dtype=np.int32)
    rc = _native.lib().pycd_hop_neighbors(
        _native.context(), *[a for x in ((pos, n), (idx, n), (idx, n))
                             for a in (x[0].ctypes.data, x[1])],
        cell.ctypes.data, pbc.ctypes.data, lo.ctypes.data, hi.ctypes.data, 1,
        1, count.ctypes.data, index.ctypes.data, vec.ctypes.data)
    assert rc == -1
    return count.ravel()


def test_every_call_of_every_thread_completes():
    """Four threads, 15 calls each, and refused ones in one of them (the
    message of a refusal is the context's, not a thread's): all of them
    return, with the numbers of the same call alone; an exception in a thread
    is the test's."""
    work = [(_table, 1), (_lists, 300), (_table, 500), (_lists, 64),
            (_table, 129)]
    alone = [f(n) for f, n in work]

    def run(first):
        done = 0
        for k in range(3 * len(work)):
            i = (first + k) % len(work)
            f, n = work[i]
            assert np.array_equal(f(n), alone[i]), work[i]
            if first == 0:
                assert (_too_full(200) == 200).all()
            done += 1
        return done

    with ThreadPoolExecutor(4) as pool:
        done = [t.result() for t in [pool.submit(run, k) for k in range(4)]]
    assert done == [3 * len(work)] * 4
