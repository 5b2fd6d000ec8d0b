"""HIP MSD kernel at the edges of its blocks, windows and parts."""
import numpy as np
import pytest

from oracle import msd as omsd
from pycd_amd import _native

pytestmark = pytest.mark.gpu

# (trajectories, path rows, carriers, lags): lag counts about the blocks of
# 64, 128 and 256 and the passes of 2 blocks; rows about a segment's origins
# (its window is 1024 rows); few paths (their origins shared by several
# workgroups) and more than 2048 (one workgroup each)
SHAPES = [(1, 1, 1, 1), (1, 2, 1, 2), (2, 5, 3, 5), (1, 70, 2, 63),
          (1, 70, 2, 64), (1, 129, 1, 65), (3, 300, 2, 127), (1, 300, 5, 128),
          (1, 700, 1, 129), (2, 1100, 3, 250), (1, 1500, 1, 256),
          (1, 900, 2, 257), (1, 1023, 1, 400), (1, 2100, 2, 512),
          (1, 2600, 1, 513), (1, 1400, 3, 1300), (1, 60, 2100, 50),
          (67, 40, 33, 40), (2, 3000, 65, 3)]


@pytest.mark.parametrize("n_traj,P,nc,M", SHAPES)
def test_shapes_against_the_oracle(n_traj, P, nc, M):
    """Each mean is a sum of at most P <= 3000 non-negative terms over the
    same differences as the oracle's: 3000 roundings of 1.1e-16 relative
    bound the difference by 3.3e-13 on either side."""
    rng = np.random.default_rng(P + M)
    pos = np.cumsum(rng.normal(size=(n_traj, P, nc, 3)), axis=1)
    ref = omsd.squared_displacement(pos.reshape(n_traj * P, nc, 3), n_traj, P,
                                    M)
    got = _native.msd(pos, M)
    assert np.allclose(got, ref, rtol=1e-12, atol=0)
    assert np.all(got[:, 0, :] == 0)


def test_non_finite_rows_stay_where_they_are():
    """A row of NaN and one of inf make exactly the means NaN or inf that
    include them, as the plain sums do."""
    rng = np.random.default_rng(3)
    pos = np.cumsum(rng.normal(size=(1, 90, 2, 3)), axis=1)
    pos[0, 80, 0, 1] = np.nan
    pos[0, 3, 1, 2] = np.inf
    with np.errstate(invalid="ignore"):
        ref = omsd.squared_displacement(pos.reshape(90, 2, 3), 1, 90, 90)
    got = _native.msd(pos, 90)
    assert np.array_equal(np.isnan(got[:, 1:]), np.isnan(ref[:, 1:]))
    fine = np.isfinite(ref)
    assert fine[0, 1:, :].any() and not fine[0, 1:, :].all()
    assert np.allclose(got[fine], ref[fine], rtol=1e-12, atol=0)
