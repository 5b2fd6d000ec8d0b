"""The plain path's hop kernel: many slots, and hops that span many path
rows."""
import random

import numpy as np
import pytest

from oracle import kmc
from pycd_amd import _native, rng

pytestmark = pytest.mark.gpu


def _runs(nc, z, rows, rows_per_hop, hops, chunk):
    """A random lattice of z slots a site (entries and energies within a few
    kT, so that many processes compete): device run and oracle's."""
    g = np.random.default_rng(100 * nc + z)
    n = 300
    a = g.normal(size=(n, n)) * 2e-4
    site = np.array([g.choice(n, size=z, replace=False) for _ in range(n)],
                    dtype=np.int32)
    lam = g.uniform(0.03, 0.04, size=(n, z))
    vab = g.uniform(0.001, 0.004, size=(n, z))
    e = g.normal(size=n) * 1e-3
    q = g.choice([-1.0, 1.0, 0.7], size=nc)
    nu, kT = 4e-4, 1.2e-3
    # the mean rate of a process, Boltzmann-weighted over its spread
    k = nu * np.exp(-(lam / 4 - vab) / kT).mean()
    args = (a + a.T, g.choice([3.0, -2.0], size=n),
            np.full(n, z, dtype=np.int32), site, g.normal(size=(n, z, 3)),
            lam, vab, e, q, np.array([1e-6, -2e-6, 5e-7]), nu, kT,
            1.0 / (nc * z * k) / rows_per_hop, rows)
    occ = [int(v) for v in g.choice(n, size=nc, replace=True)]
    gen = random.Random(7)
    state = gen.getstate()
    ora = kmc.run(kmc.Problem(*args), list(occ), gen.random, max_hops=hops,
                  record=True)
    sess = _native.KmcSession(_native.KmcProblem(*args), chunk=chunk)
    gpu = sess.run(occ, rng.UniformStream(state), max_hops=hops, record=True)
    sess.close()
    return gpu, ora


def _same(gpu, ora):
    """Same events and rows; dG0 (the reference's dot over 300 sites carries
    about 2e-15 Ha), clock and energies as in the other tests of the loop."""
    assert np.array_equal(gpu["procs"], ora["procs"])
    assert gpu["start"] == ora["start"]
    t, tr = gpu["time_data"][1:], ora["time_data"][1:]
    assert np.max(np.abs(t - tr) / tr) < 5e-12
    assert np.max(np.abs(gpu["unwrapped"] - ora["unwrapped"])) < 1e-8
    assert np.max(np.abs(gpu["delg_0"] - ora["delg_0"])) < 1e-13
    scale = max(1.0, np.max(np.abs(ora["energy"])))
    assert np.max(np.abs(gpu["energy"] - ora["energy"])) < 1e-10 * scale
    assert np.allclose(gpu["drift"], ora["drift"], rtol=1e-9, atol=0)


@pytest.mark.parametrize("nc,z", [
    (1, 13), (1, 16),  # four helpers; the widest look-ahead with four
    (5, 17),           # five, none
    (3, 33), (1, 61),  # helpers beyond the slots' groups of four, and all 14
    (9, 64),           # as many as the process wavefronts leave room for
    (42, 13), (35, 16),  # look-aheads that take the block past 64 KiB of LDS
    (30, 17), (121, 4),  # the most carriers, none and one
])
def test_helpers_of_many_slots(nc, z):
    gpu, ora = _runs(nc, z, 2001, 1.0, 200, 97)
    _same(gpu, ora)


@pytest.mark.parametrize("rows_per_hop", [2.0, 300.0])
@pytest.mark.parametrize("nc,z", [(1, 1), (1, 16), (2, 4), (3, 8), (7, 5),
                                  (22, 3), (31, 2), (32, 2), (33, 2),
                                  (70, 1)])
def test_hops_over_many_rows(nc, z, rows_per_hop):
    """1 to 32 carriers share a wavefront's lanes between path rows, more do
    not; hops of none to a few rows, and of hundreds."""
    gpu, ora = _runs(nc, z, 9001, rows_per_hop, 60, 13)
    assert gpu["start"] > 60
    _same(gpu, ora)
