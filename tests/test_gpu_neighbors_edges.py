"""Neighbour lists at the edges of the 64-target sweep, against NumPy."""
import itertools

import numpy as np
import pytest

from pycd_amd import _native

pytestmark = pytest.mark.gpu

CELL = np.array([[9.0, 0.4, -0.7], [-4.1, 8.2, 0.3], [0.9, -0.5, 12.0]])


def _images(d, pbc):
    """Minimum-image vectors of the differences d (PyCD/core.py:304-361)."""
    f = d @ np.linalg.inv(CELL)
    f -= np.where(pbc, np.round(f), 0.0)
    best = f @ CELL
    for o in itertools.product((-1, 0, 1), repeat=3):
        v = (f + np.where(pbc, o, 0)) @ CELL
        near = (v * v).sum(-1) < (best * best).sum(-1)
        best = np.where(near[..., None], v, best)
    return best


@pytest.mark.parametrize("windows", [
    [(0.0, 2.0)], [(1.0, 3.0), (0.0, 2.5), (2.9, 3.1)],
    [(-2.0, 40.0)],             # every target, the centre itself included
    [(3.0, 1.0), (-2.0, -1.0)], # nothing
])
@pytest.mark.parametrize("pbc", [[1, 1, 1], [1, 0, 1], [0, 0, 0]])
@pytest.mark.parametrize("n,n_centers", [(1, 1), (63, 7), (64, 8), (65, 9),
                                         (333, 40)])
def test_lists_against_numpy(n, n_centers, pbc, windows):
    """Sites in and around the cell, centres and targets in the caller's
    order.  The vectors are sums of three products of numbers up to a few
    tens, through an inverse of condition ~3: 1e-11 bounds their rounding."""
    g = np.random.default_rng(n)
    pos = g.uniform(-1.3, 1.7, size=(n, 3)) @ CELL
    centers = g.permutation(n)[:n_centers]
    targets = g.permutation(n)
    count, index, vec = _native.hop_neighbors(
        pos, centers, targets, CELL, pbc, [a for a, _ in windows],
        [b for _, b in windows], max_per=max(4, n))
    v = _images(pos[targets][None] - pos[centers][:, None],
                np.array(pbc, dtype=bool))
    r = np.sqrt((v * v).sum(-1))
    for s, (lo, hi) in enumerate(windows):
        for c in range(len(centers)):
            hits = np.flatnonzero((lo < r[c]) & (r[c] <= hi))
            assert count[c, s] == len(hits)
            assert np.array_equal(index[c, s, :len(hits)], hits)
            if len(hits):
                assert np.max(np.abs(vec[c, s, :len(hits)]
                                     - v[c, hits])) < 1e-11


@pytest.mark.parametrize("n_centers", [6143, 6145, 16383, 16384, 16387])
def test_centres_per_wavefront(n_centers):
    """The numbers of centres around which a wavefront takes one, two or
    four of them, with remainders; sites serve as centres many times over.
    Bound on the vectors as above."""
    n, lo, hi = 70, [0.5, 0.0], [3.0, 2.0]
    g = np.random.default_rng(n_centers)
    pos = g.uniform(-0.5, 1.5, size=(n, 3)) @ CELL
    centers = g.integers(0, n, size=n_centers)
    targets = g.permutation(n)
    count, index, vec = _native.hop_neighbors(
        pos, centers, targets, CELL, [1, 1, 1], lo, hi, max_per=n)
    v = _images(pos[targets][None] - pos[:, None], np.ones(3, dtype=bool))
    r = np.sqrt((v * v).sum(-1))
    for c in range(n):
        rows = np.flatnonzero(centers == c)
        for s in range(2):
            hits = np.flatnonzero((lo[s] < r[c]) & (r[c] <= hi[s]))
            assert (count[rows, s] == len(hits)).all()
            assert (index[rows, s, :len(hits)] == hits).all()
            if len(hits):
                assert np.max(np.abs(vec[rows, s, :len(hits)]
                                     - v[c, hits])) < 1e-11
