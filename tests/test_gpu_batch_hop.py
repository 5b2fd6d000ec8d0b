"""The batched hop loop at every processes-per-lane count and slot count,
against the oracle."""
import random

import numpy as np
import pytest

from oracle import kmc, seeding
from pycd_amd import batch as B, rng

pytestmark = pytest.mark.gpu

CELLS, NU = (5, 4, 3), 2


def _lattice(z, seed):
    """A periodic lattice of random entries, slots and hop vectors (Family
    and the full arrays the oracle reads)."""
    g = np.random.default_rng(seed)
    idx = np.stack(np.meshgrid(*[np.arange(n) for n in CELLS], np.arange(NU),
                               indexing="ij"), -1).reshape(-1, 4)
    n = len(idx)

    def site(cell, sub):
        c = np.mod(cell, CELLS)
        return ((c[..., 0] * CELLS[1] + c[..., 1]) * CELLS[2]
                + c[..., 2]) * NU + sub

    row = g.normal(size=(NU, n)) * 2e-4
    shifted = site(idx[None, :, :3] - idx[:, None, :3], idx[None, :, 3])
    table = row[idx[:, 3][:, None], shifted]
    table = table + table.T
    f = B.Family.__new__(B.Family)
    f.run, f.cells, f.n_unit, f.n_sites, f.z = None, list(CELLS), NU, n, z
    f.table = np.ascontiguousarray(table[:NU])
    f.lattice_q = np.ascontiguousarray(np.array([3.0, -2.0])[idx[:, 3]])
    slots = [g.choice(n, size=z, replace=False) for _ in range(NU)]
    order = [g.permutation(z) for _ in range(n)]
    pick = np.array([[slots[s][k] for k in o]
                     for s, o in zip(idx[:, 3], order)])
    f.nbr_site = np.ascontiguousarray(
        site(idx[pick][:, :, :3] + idx[:, None, :3], idx[pick][:, :, 3]),
        dtype=np.int32)

    def per_slot(v):
        return np.ascontiguousarray(
            [v[s][o] for s, o in zip(idx[:, 3], order)])

    f.nbr_vec = per_slot(g.normal(size=(NU, z, 3)))
    f.nbr_lambda = per_slot(g.uniform(0.03, 0.04, size=(NU, z)))
    f.nbr_vab = per_slot(g.uniform(0.001, 0.004, size=(NU, z)))
    f.site_energy = np.ascontiguousarray((g.normal(size=NU) * 1e-3)[idx[:, 3]])
    f.hop_sites = list(range(n))
    f.nu, f.volume, f.alpha = 4e-4, 1.0, 1.0
    return f, table


@pytest.mark.parametrize("z,counts", [
    (4, [1, 16, 17, 33, 48, 64]),  # 1 to 4 processes per lane
    (1, [15, 31, 49, 64]),
    (5, [25, 51, 52]),             # a second round of new slots
    (7, [1, 18, 36, 64]),          # up to 7 processes per lane
])
def test_batch_hops_vs_oracle(z, counts):
    fam, table = _lattice(z, z)
    hops, seed, kT = 300, 5, 1.2e-3
    field = np.array([1e-6, -2e-6, 5e-7])
    occs, words = rng.seeded_starts(seed, len(counts),
                                    [fam.hop_sites] * len(counts), counts)
    trajs = [dict(family=0, n_carriers=c, carrier_q=-1.0, field=field, kT=kT,
                  time_interval=1e5 / c, ewald_neut=0.0, n_path=4001,
                  max_hops=hops) for c in counts]
    out = {}
    for rates in ("f64", "f32"):
        for diff in (True, False):
            bt = B.KmcBatch([fam], "f64", rates)
            bt.set_hop_differences(diff)
            bt.setup(trajs, occs, words)
            bt.run()
            out[rates, diff] = (bt.results(),
                                [bt.rows(k) for k in range(len(counts))])
            bt.close()
    for k, c in enumerate(counts):
        pb = kmc.Problem(table, fam.lattice_q, np.full(fam.n_sites, z),
                         fam.nbr_site, fam.nbr_vec, fam.nbr_lambda,
                         fam.nbr_vab, fam.site_energy, np.full(c, -1.0), field,
                         fam.nu, kT, trajs[k]["time_interval"], 4001)
        gen = random.Random()
        gen.setstate(seeding.trajectory_states(seed, len(counts))[k])
        occ = seeding.initial_occupancy(gen, fam.hop_sites, c)
        ora = kmc.run(pb, occ, gen.random, max_hops=hops)
        for (rates, diff), (res, rows) in out.items():
            # FP32 rates: the exponent gs / kT (up to ~10) carries FP32
            # roundings, about 1e-6 of a rate and so of the clock
            tol = 1e-12 if rates == "f64" else 1e-5
            assert res["hops"][k] == ora["hops"], (rates, diff, c)
            assert abs(res["t"][k] - ora["time_data"][-1]) <= \
                tol * ora["time_data"][-1], (rates, diff, c)
            if rates == "f64":
                assert res["start"][k] == ora["start"]
                assert np.max(np.abs(rows[k] - ora["unwrapped"])) < 1e-8
            scale = max(1.0, abs(ora["energy_now"]))
            assert abs(res["energy"][k] - ora["energy_now"]) < 1e-9 * scale
            drift = np.max(np.abs(ora["drift"]))
            assert np.allclose(res["drift"][k, :c], ora["drift"],
                               rtol=max(1e-9, tol), atol=drift * max(1e-12, tol))
