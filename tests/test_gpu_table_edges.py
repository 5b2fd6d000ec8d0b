"""HIP FP64 Ewald table at the edges of its tiles, against the oracle."""
import numpy as np
import pytest

from oracle import ewald
from pycd_amd import _native

pytestmark = pytest.mark.gpu

# A triclinic cell (bohr) with one site per ~60 bohr^3, no symmetry.
CELL = np.array([[1.0, 0.07, -0.11], [-0.21, 1.1, 0.05], [0.13, 0.02, 0.9]])


def _case(n, seed=11):
    rng = np.random.default_rng(seed + n)
    cell = CELL * (60.0 * max(n, 20)) ** (1 / 3)
    return rng.uniform(size=(n, 3)) @ cell, cell


@pytest.mark.parametrize("variant", [1, 2])
@pytest.mark.parametrize("pbc", [[1, 1, 1], [1, 0, 1]])
@pytest.mark.parametrize("n", [1, 2, 15, 17, 63, 64, 65, 127, 128, 129, 193,
                               321, 1025])
def test_edge_sizes_against_the_oracle(n, pbc, variant):
    """Sizes about the edges of the 64 and 128 tiles and their 16-blocks;
    one k vector count that fills no slice; a cutoff that keeps some pairs
    and drops others.  An entry is a sum of 2 K <= 600 products of size
    2/eps w_k <= max|A|, so 600 ulp (1.3e-13) bounds its rounding; 1e-12 of
    the table's scale is the bar of every table test."""
    pos, cell = _case(n)
    alpha, r_cut, eps = 0.09, 9.0, 2.5
    k_cut = 2.1 * 2 * np.pi / np.linalg.norm(cell[0])
    rows = sorted({0, n // 2, n - 1})
    ref = ewald.table_rows(pos, rows, cell, np.ones(3, dtype=int), pbc, alpha,
                           r_cut, k_cut, eps)
    try:
        _native.set_table_variant("f64", variant)
        got, rep = _native.pair_table(pos, cell, cell, pbc, alpha, r_cut,
                                      k_cut, eps)
        none, rep0 = _native.pair_table(pos, cell, cell, pbc, alpha, r_cut,
                                        0.0, eps)
    finally:
        _native.set_table_variant("f64", 0)
    assert rep["n_kvec"] > 0 and rep0["n_kvec"] == 0
    assert rep["n_real_pairs"] == rep0["n_real_pairs"] >= n
    scale = np.max(np.abs(got))
    assert np.max(np.abs(got[rows] - ref)) <= 1e-12 * scale
    assert np.array_equal(got, got.T)
    # without a k vector: the real-space and self terms alone
    near = none != 0.0
    assert near.sum() == rep0["n_real_pairs"]


@pytest.mark.parametrize("n,k_cells", [(1, 9.1), (65, 9.1), (129, 7.3),
                                       (1408, 3.1), (1472, 3.1)])
def test_column_parts_against_the_oracle(n, k_cells):
    """Small tables are contracted in parts of the columns of Y: as many as
    the CUs take (129 sites: 50 of them), two for 22 tiles of 64 a side, one
    for 23.  A sum of 2 K <= 6000 products carries at most 6000 half ulp in
    any order, 7e-13 of the table's scale: within the 1e-12 of every table
    test.  Tile variants share the parts and give the same table."""
    pos, cell = _case(n)
    alpha, r_cut, eps = 0.09, 9.0, 2.5
    k_cut = k_cells * 2 * np.pi / np.linalg.norm(cell[0])
    rows = sorted({0, n // 2, n - 1})
    ref = ewald.table_rows(pos, rows, cell, np.ones(3, dtype=int), [1, 1, 1],
                           alpha, r_cut, k_cut, eps)
    got = {}
    try:
        for v in (1, 2):
            _native.set_table_variant("f64", v)
            got[v], rep = _native.pair_table(pos, cell, cell, [1, 1, 1], alpha,
                                             r_cut, k_cut, eps)
    finally:
        _native.set_table_variant("f64", 0)
    assert rep["n_kvec"] <= 3000
    assert np.array_equal(got[1], got[2])
    assert np.array_equal(got[1], got[1].T)
    assert np.max(np.abs(got[1][rows] - ref)) <= 1e-12 * np.max(np.abs(got[1]))
