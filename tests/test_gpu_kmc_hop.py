"""The plain path's hop kernel over its range of carriers and slots, against
the oracle."""
import random

import numpy as np
import pytest

from oracle import kmc
from pycd_amd import _native, rng, workloads
from tests.kmc_helpers import native_problem, run_gpu, run_oracle

pytestmark = pytest.mark.gpu


def _same_run(gpu, ora, hops):
    """Same events; rows, dG0 and energies as the plain path's other tests
    hold them.  The reference's dot over the sites carries about 2e-15 Ha
    into a dG0, 2e-12 of its rate at kT = 1e-3 Ha; the clock adds up the
    inverse of their sum: 5e-12 relative bounds it with the roundings of up
    to 576 rates beside."""
    assert gpu["hops"] == hops
    assert np.array_equal(gpu["procs"], ora["procs"])
    t, tr = gpu["time_data"][1:], ora["time_data"][1:]
    assert np.max(np.abs(t - tr) / tr) < 5e-12
    assert np.max(np.abs(gpu["unwrapped"] - ora["unwrapped"])) < 1e-8
    assert np.max(np.abs(gpu["delg_0"] - ora["delg_0"])) < 1e-13
    scale = max(1.0, np.max(np.abs(ora["energy"])))
    assert np.max(np.abs(gpu["energy"] - ora["energy"])) < 1e-10 * scale
    assert np.allclose(gpu["drift"], ora["drift"], rtol=1e-9, atol=0)


@pytest.mark.parametrize("edge,nc,field,compact", [
    (4, 64, 1e6, True),    # a 768-site table, read whole
    (6, 65, 0.0, True),    # cell-0 rows, two carriers in a lane
    (6, 100, 1e7, False),  # full table
    (5, 121, 1e6, False),  # the most carriers that 4 slots allow
])
def test_many_carriers_vs_oracle(edge, nc, field, compact):
    w = workloads.corundum(edge, n_carriers=nc, field_vpm=field,
                           t_final=1e-9, time_interval=1e-14)
    table = w.build_table()
    run = w.make_run(table)
    n = 400
    sess = _native.KmcSession(native_problem(run, table, compact))
    assert sess.variant() == "workgroup"
    gpu, _ = run_gpu(run, table, 2, nc, max_hops=n, session=sess, chunk=257)
    sess.close()
    _same_run(gpu, run_oracle(run, table, 2, nc, max_hops=n), n)


@pytest.mark.parametrize("nc,z,max_z", [
    (1, 1, 1),     # one process
    (1, 64, 64),   # one carrier, all processes at one site
    (17, 3, 3),    # a second carrier in a lane of the fresh sums
    (32, 8, 8),    # two helpers' fresh rows in one turn
    (300, 1, 1),   # carriers past 128: the fresh sums' general part
    (64, 5, 6),    # slot tables wider than the slots
    (30, 11, 11),  # fresh rows in two helpers' turns
    (14, 13, 13),  # the widest look-ahead
    (14, 14, 15),  # none
    (14, 22, 22),
    (14, 23, 24),
    (9, 64, 64),   # 576 processes: two per thread
])
def test_random_lattices_vs_oracle(nc, z, max_z):
    """Random tables, slots and charges: any z up to 64, any n_c that fits.
    Entries and energies keep dG0 within a few kT, so that many processes
    compete."""
    g = np.random.default_rng(nc + z)
    n, hops = 400, 300
    a = g.normal(size=(n, n)) * 2e-4
    table = a + a.T
    site = np.full((n, max_z), -1, dtype=np.int32)
    for s in range(n):
        site[s, :z] = g.choice(n, size=z, replace=False)
    vec = g.normal(size=(n, max_z, 3))
    lam = g.uniform(0.03, 0.04, size=(n, max_z))
    vab = g.uniform(0.001, 0.004, size=(n, max_z))
    e = g.normal(size=n) * 1e-3
    q_lat = g.choice([3.0, -2.0], size=n)
    q = g.choice([-1.0, 1.0, 0.7], size=nc)
    field = np.array([1e-6, -2e-6, 5e-7])
    nu, kT, P = 4e-4, 1.2e-3, 301
    rate = nc * z * nu * np.exp(-0.006 / kT)
    dt = 4 * hops / rate / P
    count = np.full(n, z, dtype=np.int32)
    args = (table, q_lat, count, site, vec, lam, vab, e, q, field, nu, kT, dt,
            P)
    occ = [int(v) for v in g.choice(n, size=nc, replace=True)]
    gen = random.Random(7)
    state = gen.getstate()
    ora = kmc.run(kmc.Problem(*args), list(occ), gen.random, max_hops=hops,
                  record=True)
    sess = _native.KmcSession(_native.KmcProblem(*args), chunk=97)
    gpu = sess.run(occ, rng.UniformStream(state), max_hops=hops, record=True)
    sess.close()
    # (some of these end on a full path)
    _same_run(gpu, ora, len(ora["procs"]))
