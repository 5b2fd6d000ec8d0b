"""HIP FP32 and BF16x3 Ewald tables at the edges of their tiles, against the
oracle and the FP64 table."""
import numpy as np
import pytest

from oracle import ewald
from pycd_amd import _native
from tests.test_gpu_table_edges import _case

pytestmark = pytest.mark.gpu

ALPHA, R_CUT, EPS = 0.09, 9.0, 2.5
# of max|A|, as in the tests of the modes on periodic lattices
TOL = {"f32": 1e-5, "bf16x3": 1e-4}


def _table(pos, cell, pbc, k_cut, mode, variant=0):
    try:
        _native.set_table_variant(mode, variant)
        return _native.pair_table(pos, cell, cell, pbc, ALPHA, R_CUT, k_cut,
                                  EPS, mode)
    finally:
        _native.set_table_variant(mode, 0)


@pytest.mark.parametrize("mode,variants", [("f32", (0,)),
                                           ("bf16x3", (1, 2, 3, 4))])
@pytest.mark.parametrize("pbc", [[1, 1, 1], [1, 0, 1]])
@pytest.mark.parametrize("n", [1, 2, 17, 63, 64, 65, 127, 128, 129, 193, 255,
                               256, 257, 385, 513])
def test_edge_sizes(n, pbc, mode, variants):
    """Sizes about the edges of the 64, 128 and 256 tiles; k vectors that
    fill no slice, and none (then only the real-space and self terms are
    left, which are FP64: the FP64 table's bits).  Off the tiles on the
    diagonal an entry's mirror is a copy; BF16x3 kernels give the same
    bits."""
    pos, cell = _case(n)
    k_cut = 2.1 * 2 * np.pi / np.linalg.norm(cell[0])
    rows = sorted({0, n // 2, n - 1})
    ref = ewald.table_rows(pos, rows, cell, np.ones(3, dtype=int), pbc, ALPHA,
                           R_CUT, k_cut, EPS)
    bare, rep0 = _table(pos, cell, pbc, 0.0, "f64")
    full, rep = _table(pos, cell, pbc, k_cut, "f64")
    scale = np.max(np.abs(full))
    block = np.arange(n) // 128
    off = block[:, None] != block[None, :]
    first = None
    for v in variants:
        none, got0 = _table(pos, cell, pbc, 0.0, mode, v)
        assert np.array_equal(none, bare), v
        got, got_rep = _table(pos, cell, pbc, k_cut, mode, v)
        for key in ("n_kvec", "n_real_pairs"):
            assert got0[key] == rep0[key] and got_rep[key] == rep[key]
        assert np.max(np.abs(got[rows] - ref)) <= TOL[mode] * scale
        assert np.max(np.abs(got - full)) <= TOL[mode] * scale
        assert np.array_equal(got[off], got.T[off])
        assert np.max(np.abs(got - got.T)) <= 1e-6 * scale
        first = got if first is None else first
        assert np.array_equal(got, first), v


@pytest.mark.parametrize("mode,n", [("f32", 2047), ("f32", 2432),
                                    ("f64", 2432), ("f32", 6080),
                                    ("f64", 6400), ("bf16x3", 4095)])
def test_sizes_about_the_choice_of_kernel(mode, n):
    """One site fewer than, as many as and one more than where the default
    kernel changes: the entries of the sites in common are the same bits."""
    pos, cell = _case(n + 2)
    k_cut = 3.1 * 2 * np.pi / np.linalg.norm(cell[0])
    small, _ = _table(pos[:n], cell, [1, 1, 1], k_cut, mode)
    for more in (1, 2):
        big, _ = _table(pos[:n + more], cell, [1, 1, 1], k_cut, mode)
        assert np.array_equal(big[:n, :n], small)
        del big
