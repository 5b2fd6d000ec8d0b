"""Performance cases: the calls that a user of this package makes, from the
smallest to the largest sizes they are made at.

  table     the Ewald pair table of one supercell (`pycd_pair_table`), in
            FP64 (the drop-in), on FP32 MFMA and on BF16x3 MFMA
  neighbors the hop neighbour lists of a supercell (`pycd_hop_neighbors`)
  kmc       one trajectory of the plain hop loop, from the seeded stream to
            the path arrays (`KmcSession.run`)
  msd       squared displacements of finished trajectories (`pycd_msd`)
  batch     many uneven trajectories in one launch with their MSD
            (`KmcBatch.run`, `results`, `msd`)
  serve     jobs of several sizes through the continuous-batching server
            (`KmcServer.submit`, `drain`)

`prepare` makes the inputs with plain torch and NumPy (pair tables
included, so that a hop loop's inputs do not depend on the table kernels)
and whatever handle a program keeps between calls; `run` is one pass.
"""
import ctypes as C
import math
import random

import numpy as np
import torch

from pycd_amd import _native, batch, constants, rng, serve, workloads

ANG = 1.889726124626  # bohr per angstrom, for the sites made here


def listed():
    return [
        # the reference's shipped example: hematite 2 x 2 x 1 with its own
        # Ewald parameters, the table handed to the host as the Python API
        # does it; the smallest call, host work and launches count
        dict(name="table_f64_120", kind="table", lattice="hematite", nx=2,
             ny=2, nz=1, precision="f64", alpha=0.2667, r_cut=4.618,
             k_cut=6.998, eps=9.355, device=False),
        # an ordinary supercell of the batched workload; the table stays on
        # the device for a hop loop created there
        dict(name="table_f64_2592", kind="table", lattice="corundum", nx=6,
             ny=6, nz=6, precision="f64", alpha=0.18, r_cut=12.0,
             k_cut=1.247155, eps=1.0, device=True),
        # the precision configuration, 10 x 10 x 10, in its three forms (the
        # FP32 one on the 8 x 8 x 8 supercell of the plain configuration)
        dict(name="table_f64_12000", kind="table", lattice="corundum", nx=10,
             ny=10, nz=10, precision="f64", alpha=0.18, r_cut=12.0,
             k_cut=1.247155, eps=1.0, device=True),
        dict(name="table_f32_6144", kind="table", lattice="corundum", nx=8,
             ny=8, nz=8, precision="f32", alpha=0.18, r_cut=12.0,
             k_cut=1.247155, eps=1.0, device=True),
        dict(name="table_bf16x3_12000", kind="table", lattice="corundum",
             nx=10, ny=10, nz=10, precision="bf16x3", alpha=0.18, r_cut=12.0,
             k_cut=1.247155, eps=1.0, device=True),
        # both hop shells of every site, once per new supercell
        dict(name="neighbors_6144", kind="neighbors", lattice="corundum",
             nx=8, ny=8, nz=8, max_per=4),
        # one electron on 3 x 3 x 3, no field: the diffusivity run of the
        # examples; each hop is a short serial chain
        dict(name="kmc_324x1", kind="kmc", lattice="corundum", nx=3, ny=3,
             nz=3, carriers=1, hops=20000, field=0.0, temp=300.0),
        # 16 electrons in 1e6 V/m on 8 x 8 x 8: the plain configuration at
        # scale
        dict(name="kmc_6144x16", kind="kmc", lattice="corundum", nx=8, ny=8,
             nz=8, carriers=16, hops=20000, field=1.0e6, temp=300.0),
        # a high carrier concentration, past what one wavefront takes
        dict(name="kmc_2592x96", kind="kmc", lattice="corundum", nx=6, ny=6,
             nz=6, carriers=96, hops=8000, field=0.0, temp=300.0),
        # the analysis of a run: 501 lags of 10001 path rows (the examples'
        # time grid), 32 trajectories of 16 carriers on the device
        dict(name="msd_32x16", kind="msd", traj=32, rows=10001, carriers=16,
             lags=501, device=True),
        # the batched form at the benchmark's width: mixed sizes, loads,
        # fields and temperatures
        dict(name="batch_4096", kind="batch", traj=4096, hops=4000, lo=4,
             hi=7, carriers=64, rates="f32", rows=200, lags=100),
        # the serving form: a burst of jobs, sliced and refilled
        dict(name="serve_64", kind="serve", jobs=64, lo=4, hi=7, carriers=32,
             hops_lo=2000, hops_hi=20000, slice=4000),
    ]


def _log(r, lo, hi):
    return int(round(math.exp(r.uniform(math.log(lo), math.log(hi)))))


def draw(r):
    kind = r.choice(["table", "table", "table", "neighbors", "kmc", "kmc",
                     "msd", "batch", "serve"])
    if kind == "table":
        lattice = r.choice(["corundum", "monoclinic", "hematite"])
        unit = len(_LATTICES[lattice][1])
        n = _log(r, 100, 11000)
        nx, ny, nz = _shape(r, n / unit)
        n = nx * ny * nz * unit
        vol = float(abs(np.linalg.det(_LATTICES[lattice][0]))) * nx * ny * nz
        kvec = _log(r, 300, min(4500, 300 + n))
        prec = r.choice(["f64", "f64", "f64", "f32", "bf16x3"])
        return dict(kind="table", lattice=lattice, nx=nx, ny=ny, nz=nz,
                    precision=prec, alpha=round(r.uniform(0.15, 0.27), 4),
                    r_cut=round(r.uniform(4.5, 12.0), 3),
                    k_cut=round((12 * math.pi ** 2 * kvec / vol) ** (1 / 3),
                                6),
                    eps=r.choice([1.0, 9.355, 38.299]),
                    device=n > 700 or r.random() < 0.5)
    if kind == "neighbors":
        lattice = r.choice(["corundum", "monoclinic"])
        unit = len(_LATTICES[lattice][1])
        nx, ny, nz = _shape(r, _log(r, 500, 10000) / unit, least=3)
        return dict(kind="neighbors", lattice=lattice, nx=nx, ny=ny, nz=nz,
                    max_per=r.choice([4, 6, 8]))
    if kind == "kmc":
        lattice = r.choice(["corundum", "monoclinic"])
        unit = len(_LATTICES[lattice][1])
        nx, ny, nz = _shape(r, _log(r, 300, 6000) / unit, least=3)
        nc = _log(r, 1, 110)
        nc = min(nc, nx * ny * nz * unit // 4)
        return dict(kind="kmc", lattice=lattice, nx=nx, ny=ny, nz=nz,
                    carriers=nc, hops=_log(r, 2000, 20000 if nc <= 32
                                           else 6000),
                    field=r.choice([0.0, 1.0e6, 1.0e7]),
                    temp=round(r.uniform(250.0, 400.0), 1))
    if kind == "msd":
        rows = _log(r, 300, 20000)
        nc = _log(r, 1, 64)
        traj = _log(r, 1, max(1, 4000000 // (rows * nc)))
        return dict(kind="msd", traj=traj, rows=rows, carriers=nc,
                    lags=min(rows, _log(r, 50, 1000)),
                    device=r.random() < 0.7)
    if kind == "batch":
        lo = r.randint(4, 6)
        return dict(kind="batch", traj=_log(r, 16, 4000),
                    hops=_log(r, 800, 4000), lo=lo, hi=r.randint(lo, 7),
                    carriers=_log(r, 4, 64), rates=r.choice(["f32", "f64"]),
                    rows=_log(r, 50, 200), lags=_log(r, 20, 100))
    lo = r.randint(4, 7)
    return dict(kind="serve", jobs=_log(r, 4, 60), lo=lo,
                hi=r.randint(lo, 7), carriers=_log(r, 2, 32), hops_lo=1000,
                hops_hi=_log(r, 2000, 18000),
                slice=r.choice([1000, 2000, 4000]))


def _shape(r, cells, least=1):
    """nx, ny, nz near a cube of `cells` cells, odd and uneven ones too,
    never more cells than that (beyond `least` per axis)."""
    edge = max(cells, 1) ** (1 / 3)
    nx = max(least, int(round(edge * r.uniform(0.8, 1.25))))
    ny = max(least, int(round(edge * r.uniform(0.8, 1.25))))
    return nx, ny, max(least, int(cells / (nx * ny)))


# ------------------------------------------------------------------ sites --
def _corundum():
    a, c = 5.038, 13.772
    return (np.array([[a, 0.0, 0.0], [-a / 2, a * math.sqrt(3) / 2, 0.0],
                      [0.0, 0.0, c]]),
            _centred([(0, 0, z) for z in (0.3553, -0.3553, 0.8553, 0.1447)]))


def _hematite():
    x = 0.3059
    o = [(x, 0, .25), (0, x, .25), (-x, -x, .25), (-x, 0, .75), (0, -x, .75),
         (x, x, .75)]
    lat, fe = _corundum()
    return lat, np.concatenate([fe, _centred(o)])


def _centred(base):
    shifts = [(0, 0, 0), (2 / 3, 1 / 3, 1 / 3), (1 / 3, 2 / 3, 2 / 3)]
    return np.array([[(b[k] + s[k]) % 1.0 for k in range(3)]
                     for s in shifts for b in base])


def _monoclinic():
    a, b, c, beta = 7.25, 11.70, 5.09, math.radians(134.2)
    return (np.array([[a, 0.0, 0.0], [0.0, b, 0.0],
                      [c * math.cos(beta), 0.0, c * math.sin(beta)]]),
            np.array([[0.0, 0.25, 0.125], [0.0, 0.75, 0.875],
                      [0.5, 0.75, 0.125], [0.5, 0.25, 0.875]]))


_LATTICES = {"corundum": _corundum(), "hematite": _hematite(),
             "monoclinic": _monoclinic()}


def _sites(case, seed, sigma):
    """Site positions (bohr) of the supercell, cell-major, each displaced by
    a normal of `sigma` angstrom; the minimum-image cell; the translational
    matrix the reference forms (its columns scaled by the size)."""
    lat, frac = _LATTICES[case["lattice"]]
    size = np.array([case["nx"], case["ny"], case["nz"]])
    cells = np.stack(np.meshgrid(*[np.arange(n) for n in size],
                                 indexing="ij"), -1).reshape(-1, 1, 3)
    pos = ((cells + frac) @ lat).reshape(-1, 3)
    pos = pos + sigma * np.random.default_rng(seed).normal(size=pos.shape)
    return pos * ANG, lat * size[:, None] * ANG, lat * size[None, :] * ANG


# ------------------------------------------- pair table in plain torch, FP64
def _images(cell):
    """The 26 neighbouring images' offsets."""
    d = [(x, y, z) for x in (-1, 0, 1) for y in (-1, 0, 1)
         for z in (-1, 0, 1) if x or y or z]
    return np.array(d, dtype=float) @ cell


def _nearest(d, cell, want_vector):
    """Minimum image of the displacements d (..., 3): squared distances, or
    the vectors."""
    inv = torch.from_numpy(np.linalg.inv(cell)).cuda()
    f = d @ inv
    b = (f - torch.round(f)) @ torch.from_numpy(cell).cuda()
    best = (b * b).sum(-1)
    out = b.clone() if want_vector else None
    for v in _images(cell):
        x, y, z = (b[..., k] + float(v[k]) for k in range(3))
        r2 = x * x + y * y + z * z
        if want_vector:
            near = (r2 < best)[..., None]
            out = torch.where(near, torch.stack((x, y, z), -1), out)
        best = torch.minimum(best, r2)
    return out if want_vector else best


def _reciprocal(trans, k_cut):
    """Half of the reciprocal vectors below k_cut, the cell volume."""
    vol = abs(np.linalg.det(trans))
    rec = 2 * np.pi * np.linalg.inv(trans).T
    km = np.ceil(k_cut / np.linalg.norm(rec, axis=1)).astype(int)
    g = np.mgrid[-km[0]:km[0] + 1, -km[1]:km[1] + 1,
                 -km[2]:km[2] + 1].reshape(3, -1).T
    a, b, c = g.T
    g = g[(a < 0) | ((a == 0) & (b < 0)) | ((a == 0) & (b == 0) & (c < 0))]
    k = g @ rec
    return k[(k * k).sum(1) < k_cut ** 2], vol


def _half_count(case):
    _, _, trans = _sites(case, 0, 0.0)
    return len(_reciprocal(trans, case["k_cut"] / ANG)[0])


def _pair_rows(pos, rows, cell, trans, alpha, r_cut, k_cut, eps):
    """Rows [0, rows) of the pair table, and the pairs within r_cut."""
    k, vol = _reciprocal(trans, k_cut)
    x = torch.from_numpy(pos).cuda()
    kv = torch.from_numpy(k).cuda()
    k2 = (kv * kv).sum(1)
    w = torch.sqrt(2 * np.pi / vol * torch.exp(-k2 / (4 * alpha)) / k2)
    ph = x @ kv.T
    y = torch.cat((w * torch.cos(ph), w * torch.sin(ph)), 1)
    del ph
    out = (2 / eps) * (y[:rows] @ y.T)
    del y
    n, pairs = len(pos), 0
    step = max(1, (1 << 22) // n)
    for lo in range(0, rows, step):
        hi = min(rows, lo + step)
        i = torch.arange(lo, hi, device="cuda")
        r2 = _nearest(x[None] - x[lo:hi, None], cell, False)
        r2[i - lo, i] = 0.0
        r = torch.sqrt(r2)
        near = r < r_cut
        pairs += int(near.sum())
        v = torch.special.erfc(math.sqrt(alpha) * r) / 2 / eps
        v = torch.where(near, v / torch.where(r > 0, r, 1.0), 0.0)
        out[lo:hi] += v
        out[i, i] -= math.sqrt(alpha / math.pi) / eps
    return out, pairs


# ------------------------------------------------------------------ table --
def _prepare_table(case, seed):
    pos, cell, trans = _sites(case, seed, 0.02)
    s = dict(case=case, n=len(pos), pos=pos, pbc=np.ones(3, dtype=np.int32),
             cell=np.ascontiguousarray(cell), trans=np.ascontiguousarray(trans),
             alpha=case["alpha"] / ANG, r_cut=case["r_cut"] * ANG,
             k_cut=case["k_cut"] / ANG)
    if case["device"]:
        s["dpos"] = torch.from_numpy(pos).cuda()
        s["out"] = torch.empty((len(pos), len(pos)), dtype=torch.float64,
                               device="cuda")
        s["ctx"], s["lib"] = _native.context(), _native.lib()
    return s


def _run_table(s):
    case = s["case"]
    if not case["device"]:
        table, rep = _native.pair_table(
            s["pos"], s["cell"], s["trans"], s["pbc"], s["alpha"], s["r_cut"],
            s["k_cut"], case["eps"], case["precision"])
        return {"table": table, "pairs": rep["n_real_pairs"],
                "kvec": rep["n_kvec"]}
    rep = _native.EwaldReport()
    rc = s["lib"].pycd_pair_table(
        s["ctx"], s["dpos"].data_ptr(), s["n"], s["cell"].ctypes.data,
        s["trans"].ctypes.data, s["pbc"].ctypes.data, s["alpha"], s["r_cut"],
        s["k_cut"], case["eps"], _native.PREC[case["precision"]],
        s["out"].data_ptr(), C.byref(rep))
    if rc:
        raise RuntimeError(f"pycd_pair_table: {rc}")
    return {"table": s["out"], "pairs": rep.n_real_pairs, "kvec": rep.n_kvec}


def _exact_table(case, seed):
    pos, cell, trans = _sites(case, seed, 0.02)
    out, pairs = _pair_rows(pos, len(pos), cell, trans, case["alpha"] / ANG,
                            case["r_cut"] * ANG, case["k_cut"] / ANG,
                            case["eps"])
    return {"table": out, "pairs": pairs, "kvec": _half_count(case)}


# -------------------------------------------------------------- neighbours --
def _shells(lattice):
    """(lo, hi] windows of the hop shells, angstrom."""
    if lattice == "corundum":
        c = [2.971, 2.901]
    else:
        c = workloads.monoclinic_shells(*_LATTICES[lattice])
    return np.array([v - 0.002 for v in c]), np.array([v + 0.002 for v in c])


def _prepare_neighbors(case, seed):
    pos, cell, _ = _sites(case, seed, 1e-4)
    lo, hi = _shells(case["lattice"])
    sites = np.arange(len(pos))
    # the sites are asked for in an order of the caller's
    order = np.random.default_rng(seed + 1).permutation(sites)
    return dict(pos=pos, cell=cell, centers=order, targets=sites,
                pbc=np.ones(3, dtype=np.int32), lo=lo * ANG, hi=hi * ANG,
                max_per=case["max_per"])


def _run_neighbors(s):
    count, index, vec = _native.hop_neighbors(
        s["pos"], s["centers"], s["targets"], s["cell"], s["pbc"], s["lo"],
        s["hi"], max_per=s["max_per"])
    held = np.arange(index.shape[2]) < count[..., None]
    return {"count": count, "index": index[held], "vec": vec[held]}


def _exact_neighbors(case, seed):
    s = _prepare_neighbors(case, seed)
    x = torch.from_numpy(s["pos"]).cuda()
    ns = len(s["lo"])
    count = np.zeros((len(x), ns), dtype=np.int32)
    index, vec = [], []
    step = max(1, (1 << 21) // len(x))
    for a in range(0, len(x), step):
        ci = torch.from_numpy(s["centers"][a:a + step]).cuda()
        v = _nearest(x[None] - x[ci, None], s["cell"], True)
        r = torch.sqrt((v * v).sum(-1))
        hits = torch.stack([(r > float(l)) & (r <= float(h))
                            for l, h in zip(s["lo"], s["hi"])], 1)
        count[a:a + step] = hits.sum(2).cpu().numpy()
        at = hits.nonzero()
        index.append(at[:, 2].to(torch.int32))
        vec.append(v[at[:, 0], at[:, 2]])
    return {"count": count, "index": torch.cat(index), "vec": torch.cat(vec)}


# ------------------------------------------------------------ one trajectory
def _mean_rate(run, temp, nc):
    """Hops per au time of nc carriers without interaction."""
    s = run.hop_site_lists["electron"][0]
    z = int(run.nbr_count[s])
    g = run.nbr_lambda[s, :z] / 4 - run.nbr_vab[s, :z]
    return nc * float(np.sum(run.material.vn
                             * np.exp(-g / (temp * constants.K2AUTEMP))))


def _workload(lattice, size, **kw):
    params = (workloads.corundum_params() if lattice == "corundum"
              else workloads.monoclinic_params())
    return workloads.Workload(params, size, **kw)


def _lattice_rows(w, whole):
    """The supercell's pair table, or its first cell's rows."""
    pos = w.neighbors.bulk_sites.cell_coordinates
    n_unit = len(pos) // int(w.size.prod())
    lat = w.material.lattice_matrix
    # a few hundred vectors, as the batched workload's supercells have
    k_cut = (12 * math.pi ** 2 * 1050 / w.system.system_volume) ** (1 / 3)
    a, _ = _pair_rows(pos, len(pos) if whole else n_unit,
                      lat * w.size[:, None], lat * w.size[None, :],
                      w.system.alpha, w.system.r_cut, k_cut, 1.0)
    return a.cpu().numpy()


def _kmc_inputs(case, seed):
    w = _workload(case["lattice"], (case["nx"], case["ny"], case["nz"]),
                  temp=case["temp"], n_carriers=case["carriers"],
                  field_vpm=case["field"])
    table = _lattice_rows(w, True)
    run = w.make_run(table)
    nc = case["carriers"]
    # carriers at work hop slower than alone, the more the more there are:
    # a path that holds the whole run
    dt = ((40 + 20 * nc) * case["hops"] / _mean_rate(run, case["temp"], nc)
          / 4000)
    gen = random.Random(seed)
    occ = [int(v) for v in gen.sample(
        [int(v) for v in run.hop_site_lists["electron"]], nc)]
    return run, table, dt, occ, gen


def _prepare_kmc(case, seed):
    run, table, dt, occ, gen = _kmc_inputs(case, seed)
    pb = _native.KmcProblem(
        table=table, lattice_q=run.base_charge_config()[:, 0],
        nbr_count=run.nbr_count, nbr_site=run.nbr_site, nbr_vec=run.nbr_vec,
        nbr_lambda=run.nbr_lambda, nbr_vab=run.nbr_vab,
        site_energy=run.system_relative_energies,
        carrier_q=np.full(case["carriers"], -1.0), field=run.electric_field,
        nu=run.material.vn, kT=run.temp, time_interval=dt, n_path=4001,
        cells=run.system_size)
    return dict(session=_native.KmcSession(pb), occ=occ,
                state=gen.getstate(), hops=case["hops"])


_KMC_OUT = ("unwrapped", "energy", "delg_0", "drift", "time_data", "t",
            "energy_now")


def _run_kmc(s):
    res = s["session"].run(s["occ"], rng.UniformStream(s["state"]),
                           max_hops=s["hops"], record=True)
    out = {k: res[k] for k in _KMC_OUT}
    out.update(t=float(res["t"]), energy_now=float(res["energy_now"]),
               occupancy=np.array(res["occupancy"]), procs=res["procs"],
               hops=int(res["hops"]), start=int(res["start"]))
    return out


def _exact_kmc(case, seed):
    run, table, dt, occ, gen = _kmc_inputs(case, seed)
    nc, P, hops = case["carriers"], 4001, case["hops"]
    z = int(run.nbr_count[occ[0]])
    q = -1.0
    q_lat = run.base_charge_config()[:, 0]
    phi = table @ q_lat
    nbr, E = run.nbr_site[:, :z], run.system_relative_energies
    lam, vab, hop = (a[:, :z] for a in (run.nbr_lambda, run.nbr_vab,
                                        run.nbr_vec))
    half = 0.5 * hop @ run.electric_field
    kT, nu = run.temp, run.material.vn
    occ = np.array(occ)
    energy = float(q_lat @ phi + 2 * q * phi[occ].sum()
                   + q * q * table[np.ix_(occ, occ)].sum())
    t, start, disp = 0.0, 1, np.zeros((nc, 3))
    rows, epath, dpath = np.zeros((P, nc, 3)), np.zeros(P), np.zeros(P)
    epath[0] = energy
    drift, times, procs = np.zeros((nc, 3)), [0.0], []
    for _ in range(hops):
        tgt = nbr[occ]
        diff = table[tgt.ravel()[:, None], occ] - np.repeat(
            table[occ[:, None], occ], z, 0)
        d = (phi[tgt] - phi[occ][:, None]
             + q * diff.sum(1).reshape(nc, z)
             + q * (table[occ, occ][:, None] - table[occ[:, None], tgt]))
        g = 2 * q * d + E[tgt] - E[occ][:, None]
        la = lam[occ]
        k = nu * np.exp(-((la + g) ** 2 / (4 * la) - vab[occ] - half[occ])
                        / kT)
        cum = np.cumsum(k.ravel())
        u1, u2 = gen.random(), gen.random()
        p = min(int(np.searchsorted(cum, u1 * cum[-1], side="right")),
                nc * z - 1)
        c, j = divmod(p, z)
        t -= math.log(u2) / cum[-1]
        end, gp = min(int(t / dt), P), float(g[c, j])
        dpath[start:end] = gp
        v = hop[occ[c], j]
        if case["field"]:
            drift[c] += v * k[c, j]
        occ[c] = tgt[c, j]
        disp[c] += v
        energy += gp
        times.append(t)
        procs.append(p)
        if end >= start + 1:
            rows[start:end] = disp
            epath[start:end] = energy
            start = end
            if end >= P:
                break
    return {"unwrapped": rows.reshape(P, 3 * nc), "energy": epath,
            "delg_0": dpath, "drift": drift, "time_data": np.array(times),
            "t": t, "energy_now": energy, "occupancy": occ,
            "procs": np.array(procs), "hops": len(procs), "start": start}


# -------------------------------------------------------------------- msd --
def _paths(case, seed):
    """Random walks with hops of ~3 angstrom, some path steps without one."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    shape = (case["traj"], case["rows"], case["carriers"], 3)
    step = torch.randn(shape, dtype=torch.float64, device="cuda", generator=g)
    move = torch.rand(shape[:3], device="cuda", generator=g) < 0.7
    step = 1.7 * step * move[..., None]
    step[:, 0] = 0.0
    return torch.cumsum(step, 1)


def _prepare_msd(case, seed):
    pos = _paths(case, seed)
    if not case["device"]:
        return dict(case=case, pos=pos.cpu().numpy())
    sd = torch.empty((case["traj"], case["lags"], case["carriers"]),
                     dtype=torch.float64, device="cuda")
    return dict(case=case, pos=pos, sd=sd, ctx=_native.context(),
                lib=_native.lib())


def _run_msd(s):
    case = s["case"]
    if not case["device"]:
        return {"sd": _native.msd(s["pos"], case["lags"])}
    rc = s["lib"].pycd_msd(s["ctx"], s["pos"].data_ptr(), case["traj"],
                           case["rows"], case["carriers"], case["lags"],
                           s["sd"].data_ptr())
    if rc:
        raise RuntimeError(f"pycd_msd: {rc}")
    return {"sd": s["sd"]}


def _exact_msd(case, seed):
    pos = _paths(case, seed)
    P = case["rows"]
    sd = torch.zeros((case["traj"], case["lags"], case["carriers"]),
                     dtype=torch.float64, device="cuda")
    for lag in range(1, case["lags"]):
        d = pos[:, lag:] - pos[:, :P - lag]
        sd[:, lag] = (d * d).sum(-1).mean(1)
    return {"sd": sd}


# ------------------------------------------------------------------ batch --
def _prepare_batch(case, seed):
    gen = np.random.default_rng(seed)
    works = [_workload("corundum", n) for n in range(case["lo"],
                                                     case["hi"] + 1)]
    fams = []
    for w in works:
        rows = _lattice_rows(w, False)
        fams.append(batch.Family(w.make_run(rows), rows))
    n = case["traj"]
    sizes = gen.integers(0, len(fams), size=n)
    ncs = gen.integers(1, case["carriers"] + 1, size=n)
    occs, words = rng.seeded_starts(seed, n,
                                    [fams[f].hop_sites for f in sizes], ncs)
    trajs = []
    for k in range(n):
        fam = fams[sizes[k]]
        d = gen.normal(size=3)
        field = (gen.uniform(0.0, 1.0e7) * constants.VPM2AUFIELD
                 * d / np.linalg.norm(d))
        temp = gen.uniform(250.0, 400.0)
        dt = 3 * case["hops"] / _mean_rate(fam.run, temp, ncs[k])
        trajs.append(dict(family=int(sizes[k]), n_carriers=int(ncs[k]),
                          carrier_q=-1.0, field=field,
                          kT=temp * constants.K2AUTEMP,
                          time_interval=dt / case["rows"], ewald_neut=0.0,
                          n_path=4 * case["rows"] + 1,
                          max_hops=case["hops"]))
    bt = batch.KmcBatch(fams, rate_precision=case["rates"])
    bt.setup(trajs, occs, words,
             order=np.argsort(-ncs, kind="stable").astype(np.int32),
             msd_lags=[case["lags"]] * n, waves_per_cu=16)
    return dict(batch=bt)


def _run_batch(s):
    bt = s["batch"]
    bt.run(use_graph=True)
    res = bt.results()
    out = {k: res[k] for k in ("t", "energy", "hops", "start", "no_select",
                               "done", "drift")}
    out["msd"] = np.concatenate(bt.msd())
    return out


# ------------------------------------------------------------------ serve --
def _serve_family(edge):
    w = _workload("monoclinic", edge)
    rows = _lattice_rows(w, False)
    return w.make_run(rows), rows


def _prepare_serve(case, seed):
    srv = serve.KmcServer(_serve_family, n_slots=48, nc_max=32,
                          rows_capacity=1 << 24, slice_hops=case["slice"],
                          path_rows=100, msd_lags=50)
    # a server that has seen its lattice sizes
    for edge in range(case["lo"], case["hi"] + 1):
        srv.submit(serve.Job(-edge, edge, 1, 10, seed=edge))
    srv.drain()
    g = np.random.default_rng(seed)
    n_c = g.permutation(np.linspace(1, case["carriers"], case["jobs"])
                        .round().astype(int))
    jobs = []
    for k in range(case["jobs"]):
        hops = math.exp(g.uniform(math.log(case["hops_lo"]),
                                  math.log(case["hops_hi"])))
        jobs.append(dict(edge=int(g.integers(case["lo"], case["hi"] + 1)),
                         n_carriers=int(n_c[k]), hops=int(hops),
                         seed=1000 * seed + k,
                         temp=float(g.uniform(250.0, 400.0)),
                         field_vpm=float(g.uniform(0.0, 1.0e7))))
    return dict(server=srv, jobs=jobs)


def _run_serve(s):
    jobs = [serve.Job(k, **j) for k, j in enumerate(s["jobs"])]
    for j in jobs:
        s["server"].submit(j)
    s["server"].drain()
    out = {k: np.array([j.result[k] for j in jobs])
           for k in ("t", "energy", "hops", "start", "no_select")}
    out["rows"] = np.concatenate([j.result["rows"].ravel() for j in jobs])
    out["msd"] = np.concatenate([j.result["msd"] for j in jobs])
    return out


# ------------------------------------------------------------------- cases --
_PREPARE = dict(table=_prepare_table, neighbors=_prepare_neighbors,
                kmc=_prepare_kmc, msd=_prepare_msd, batch=_prepare_batch,
                serve=_prepare_serve)
_RUN = dict(table=_run_table, neighbors=_run_neighbors, kmc=_run_kmc,
            msd=_run_msd, batch=_run_batch, serve=_run_serve)
# (batched and served trajectories make their choices on FP32 rates, which a
# restatement in 64 bits does not follow event by event)
_EXACT = dict(table=_exact_table, neighbors=_exact_neighbors, kmc=_exact_kmc,
              msd=_exact_msd)


def prepare(case, seed):
    return dict(_PREPARE[case["kind"]](case, seed), kind=case["kind"])


def run(state):
    return _RUN[state["kind"]](state)


def exact(case, seed):
    f = _EXACT.get(case["kind"])
    return f(case, seed) if f else None


def _hop_work(nc, z, hops):
    """One hop: the table entries that change, (1 + z)(2 n_c - 1), the new
    processes' records, the two uniforms; a rate per process (~40
    operations) and the sums that the entries enter."""
    gathers = (1 + z) * (2 * nc - 1)
    return (hops * (8.0 * gathers + 80 * z + 16),
            hops * (40.0 * nc * z + 2 * gathers))


def work(case):
    kind = case["kind"]
    if kind in ("table", "neighbors"):
        unit = len(_LATTICES[case["lattice"]][1])
        n = unit * case["nx"] * case["ny"] * case["nz"]
    if kind == "table":
        k = 2 * _half_count(case)
        # the symmetric product, once per unordered pair (three products in
        # the BF16 split), and ~100 operations for a pair's distance
        times = 3 if case["precision"] == "bf16x3" else 1
        return {"bytes": 8.0 * n * n + 24.0 * n,
                "flops": n * (n + 1.0) * (k * times + 50)}
    if kind == "neighbors":
        shells = len(_shells(case["lattice"])[0])
        return {"bytes": 24.0 * n + 16.0 * n
                + n * shells * (4.0 + 28.0 * case["max_per"]),
                "flops": 0.5 * n * n * 30.0}
    if kind == "kmc":
        nc, z = case["carriers"], 4
        b, f = _hop_work(nc, z, case["hops"])
        return {"bytes": b + 12.0 * case["hops"] + 4001 * (24.0 * nc + 16),
                "flops": f}
    if kind == "msd":
        units = case["traj"] * case["carriers"]
        pairs = case["lags"] * (case["rows"] - 0.5 * case["lags"])
        return {"bytes": units * (24.0 * case["rows"] + 8.0 * case["lags"]),
                "flops": 8.0 * units * pairs}
    if kind == "batch":
        n, nc = case["traj"], case["carriers"] / 2
        b, f = _hop_work(nc, 4, case["hops"])
        rows = 1.5 * case["rows"]
        return {"bytes": n * (b + 24.0 * nc * rows + 8.0 * case["lags"]),
                "flops": n * (f + 6.0 * nc * case["lags"] * rows)}
    n, nc = case["jobs"], case["carriers"] / 2
    mean = ((case["hops_hi"] - case["hops_lo"])
            / math.log(case["hops_hi"] / case["hops_lo"]))
    b, f = _hop_work(nc, 4, mean)
    return {"bytes": n * (b + 24.0 * nc * 401), "flops": n * f}
