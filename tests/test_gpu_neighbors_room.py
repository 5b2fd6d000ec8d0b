"""The room past a shell's entries in the neighbour lists."""
import numpy as np
import pytest

from pycd_amd import _native

pytestmark = pytest.mark.gpu

CELL = np.array([[9.0, 0.4, -0.7], [-4.1, 8.2, 0.3], [0.9, -0.5, 12.0]])


@pytest.mark.parametrize("n,n_centers", [(1, 1), (65, 65), (130, 7),
                                         (70, 6145), (70, 13823),
                                         (70, 13824), (70, 16387)])
def test_nothing_of_an_earlier_call_is_left(n, n_centers):
    """A call with every target in its shells, then one of the same sizes
    (so in the same memory) with few or none: zeros past the counts, for
    one, two and four centres per wavefront and more than 64 entries."""
    g = np.random.default_rng(n)
    pos = g.uniform(size=(n, 3)) @ CELL
    centers = g.integers(0, n, size=n_centers)
    targets = g.permutation(n)
    for lo, hi in ([-1.0, -1.0], [40.0, 40.0]), ([0.0, 2.0], [1.5, 2.5]):
        count, index, vec = _native.hop_neighbors(
            pos, centers, targets, CELL, [1, 1, 1], lo, hi, max_per=n + 3)
        past = np.arange(n + 3) >= count[..., None]
        assert past.any() and not past.all() or lo[0] >= 0
        assert not index[past].any()
        assert not vec[past].any()
