"""The context's workspace: shared by threads, bounded, given back."""
import threading

import numpy as np
import pytest
import torch

from pycd_amd import _native

pytestmark = pytest.mark.gpu

CELL = np.diag([1.0, 1.1, 0.9])


def _table(n):
    cell = CELL * (60.0 * max(n, 20)) ** (1 / 3)
    pos = np.random.default_rng(n).uniform(size=(n, 3)) @ cell
    return _native.pair_table(pos, cell, cell, [1, 1, 1], 0.09, 9.0,
                              1.5 * 2 * np.pi / np.linalg.norm(cell[0]), 2.5)[0]


def _lists(n):
    pos = np.random.default_rng(n).uniform(size=(n, 3)) @ (20 * CELL)
    count, index, vec = _native.hop_neighbors(
        pos, np.arange(n), np.arange(n), 20 * CELL, [1, 1, 1], [0.0], [4.0],
        max_per=n)
    held = np.arange(n) < count[..., None]
    return np.concatenate([count.ravel(), index[held], vec[held].ravel()])


def test_threads_share_a_context():
    """Calls of several sizes at once give what they give one by one."""
    work = [(_table, 1), (_table, 65), (_lists, 300), (_table, 500),
            (_lists, 64), (_table, 129)]
    alone = [f(n) for f, n in work]
    wrong = []

    def run(first):
        for k in range(3 * len(work)):
            i = (first + k) % len(work)
            f, n = work[i]
            if not np.array_equal(f(n), alone[i]):
                wrong.append(work[i])

    threads = [threading.Thread(target=run, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


def test_kept_memory_is_bounded():
    """Tables of 72 to 648 MB, the last larger than what may be kept (512
    MiB): never more than that stays allocated beyond the calls."""
    _table(64)
    free = torch.cuda.mem_get_info()[0]
    for n in (3000, 4500, 6000, 7500, 9000, 4500):
        _table(n)
        kept = free - torch.cuda.mem_get_info()[0]
        assert kept <= (512 << 20) + (64 << 20), (n, kept)
