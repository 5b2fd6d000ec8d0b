"""HIP MSD calls of few paths: lags and origins shared by workgroups, and the
kernel of the smallest calls."""
import numpy as np
import pytest

from oracle import msd as omsd
from pycd_amd import _native

pytestmark = pytest.mark.gpu

# (trajectories, path rows, carriers, lags)
SHAPES = [
    # lags in passes of 128: whole ones, one lag over, one lag short; origins
    # in parts, some of which have none in the last passes
    (1, 2049, 1, 128), (1, 2049, 1, 129), (1, 2600, 1, 2600),
    (2, 2050, 3, 511), (3, 4100, 2, 513),
    # lags shared, origins not; both in groups of 64 and 32 lanes
    (7, 700, 9, 700), (8, 700, 8, 513), (65, 300, 3, 300), (4, 2100, 17, 90),
    # origins in parts of several segments (parts at their most)
    (1, 60000, 1, 20),
    # about the lines of the short kernel: rows 64 and 2048, blocks of 8 lags
    # 256 (one pass of lags) and 512, blocks times rows 450000
    (1, 64, 1, 64), (1, 65, 1, 64), (1, 65, 1, 1), (1, 2048, 1, 33),
    (1, 2048, 1, 2048), (4, 200, 8, 64), (4, 200, 8, 65), (4, 200, 8, 129),
    (16, 140, 2, 128), (16, 140, 2, 136), (3, 1700, 1, 700),
    (3, 1700, 1, 720),
    # too many paths to share
    (41, 90, 50, 90), (64, 140, 32, 129),
]


@pytest.mark.parametrize("n_traj,P,nc,M", SHAPES)
def test_shapes_against_the_oracle(n_traj, P, nc, M):
    """Each mean is a sum of at most P non-negative terms over the same
    differences as the oracle's, in chains of a few hundred roundings at most
    on the device: P roundings of 1.1e-16 on the oracle's side (its sums over
    an array are pairwise, fewer) and 500 here stay below 1e-12."""
    rng = np.random.default_rng(P + M)
    pos = np.cumsum(rng.normal(size=(n_traj, P, nc, 3)), axis=1)
    ref = omsd.squared_displacement(pos.reshape(n_traj * P, nc, 3), n_traj, P,
                                    M)
    got = _native.msd(pos, M)
    assert np.allclose(got, ref, rtol=1e-12, atol=0)
    assert np.all(got[:, 0, :] == 0)


@pytest.mark.parametrize("P,M", [(300, 300), (2100, 2100)])
def test_non_finite_rows_stay_where_they_are(P, M):
    """A row of NaN and one of inf make exactly the means NaN or inf that
    include them, in the short kernel and with lags and origins shared."""
    rng = np.random.default_rng(3)
    pos = np.cumsum(rng.normal(size=(1, P, 2, 3)), axis=1)
    pos[0, P - 10, 0, 1] = np.nan
    pos[0, 3, 1, 2] = np.inf
    with np.errstate(invalid="ignore"):
        ref = omsd.squared_displacement(pos.reshape(P, 2, 3), 1, P, M)
    got = _native.msd(pos, M)
    assert np.array_equal(np.isnan(got[:, 1:]), np.isnan(ref[:, 1:]))
    fine = np.isfinite(ref)
    assert fine[0, 1:, :].any() and not fine[0, 1:, :].all()
    assert np.allclose(got[fine], ref[fine], rtol=1e-12, atol=0)
