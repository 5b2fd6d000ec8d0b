"""Accuracy of the HIP MSD sums against extended precision."""
import numpy as np
import pytest

from pycd_amd import _native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_traj,P,nc,M", [
    (16, 2001, 16, 2001),  # groups of 64 lanes, lags shared
    (4, 1000, 32, 1000),   # groups of 64 lanes, many sums of few origins
    (8, 600, 16, 600),     # of 32
])
def test_sums_are_as_exact_as_pairwise_ones(n_traj, P, nc, M):
    """The device's sums and NumPy's pairwise ones of the same differences
    end in the same two roundings (the sum's and the mean's); the levels of
    the sums on either side keep what comes before below those.  Over all
    lags of four paths the device's 2-norm error is NumPy's within a quarter
    (the spread of either between paths is a tenth)."""
    pos = np.cumsum(np.random.default_rng(1).normal(size=(n_traj, P, nc, 3)),
                    axis=1)
    got = _native.msd(pos, M)
    dev = ref = 0.0
    for c in range(4):
        p = pos[0, :, c]
        e = p.astype(np.longdouble)
        err = np.zeros((3, M))
        for tau in range(1, M):
            d = e[tau:] - e[:P - tau]
            exact = (d * d).sum() / (P - tau)
            d = p[tau:] - p[:P - tau]
            plain = np.mean(np.einsum("ij,ij->i", d, d))
            err[:, tau] = got[0, tau, c] - exact, plain - exact, exact
        dev += np.linalg.norm(err[0]) / np.linalg.norm(err[2])
        ref += np.linalg.norm(err[1]) / np.linalg.norm(err[2])
    assert dev <= 1.25 * ref, (dev / 4, ref / 4)
