"""Tables about the sizes where the blocks that finish an entry change."""
import numpy as np
import pytest

from oracle import ewald
from pycd_amd import _native
from tests.test_gpu_table_edges import _case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode,tol", [("f64", 1e-12), ("f32", 1e-5)])
@pytest.mark.parametrize("n", [960, 961])
def test_rows_of_the_finish_blocks(n, mode, tol):
    """15 and 16 tiles of 64 a side (blocks of 16 and of 64 rows): rows of
    the first, a middle and the last tile against the oracle, the mirror a
    copy, the ordered pairs within the cutoff counted once each."""
    pos, cell = _case(n)
    k_cut = 2.1 * 2 * np.pi / np.linalg.norm(cell[0])
    rows = [0, 15, 16, 63, 64, n // 2, n - 2, n - 1]
    ref = ewald.table_rows(pos, rows, cell, np.ones(3, dtype=int), [1, 1, 0],
                           0.09, 9.0, k_cut, 2.5)
    got, rep = _native.pair_table(pos, cell, cell, [1, 1, 0], 0.09, 9.0,
                                  k_cut, 2.5, mode)
    bare, rep0 = _native.pair_table(pos, cell, cell, [1, 1, 0], 0.09, 9.0,
                                    0.0, 2.5, mode)
    assert np.max(np.abs(got[rows] - ref)) <= tol * np.max(np.abs(got))
    assert np.array_equal(got, got.T)
    assert (bare != 0.0).sum() == rep0["n_real_pairs"] == rep["n_real_pairs"]
