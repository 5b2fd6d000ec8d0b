"""The forms of the plain path's hop kernel that differ: cell-0 rows and the
full table, a trajectory in one launch and in many, against the oracle event
for event."""
import numpy as np
import pytest

from pycd_amd import _native, rng, workloads
from tests.kmc_helpers import native_problem, run_oracle, seeded_start

pytestmark = pytest.mark.gpu

KEYS = ("procs", "time_data", "unwrapped", "energy", "delg_0", "drift")


def _run(run, table, nc, hops, compact, chunk):
    sess = _native.KmcSession(native_problem(run, table, compact),
                              chunk=chunk, max_chunk=chunk)
    n_unit = len(table) // int(np.prod(run.system_size))
    assert sess.table_rows() == (n_unit if compact else len(table))
    gen, occ = seeded_start(run, 2, nc)
    res = sess.run(occ, rng.UniformStream(gen.getstate()), max_hops=hops,
                   record=True)
    sess.close()
    return res


@pytest.mark.parametrize("nc", [1, 16, 48, 90])
def test_forms_give_the_oracles_events(nc):
    """6 x 6 x 6 corundum (2592 sites, a 54 MB table, above which cell-0 rows
    are read) in 1e6 V/m: the oracle's events in each form.  Launches of any
    length leave the same numbers: what a launch begins with is formed from
    the state, correctly rounded, as what hops keep up is.  Cell-0 rows equal
    the table's to 1e-14 of its scale, so the clock to 1e-11."""
    w = workloads.corundum(6, n_carriers=nc, field_vpm=1e6, t_final=1e-9,
                           time_interval=1e-14)
    table = w.build_table()
    run = w.make_run(table)
    hops = 600
    ora = run_oracle(run, table, 2, nc, max_hops=hops)
    for compact in (True, False):
        whole = _run(run, table, nc, hops, compact, 4096)
        assert whole["hops"] == hops
        assert np.array_equal(whole["procs"], ora["procs"])
        t, tr = whole["time_data"][1:], ora["time_data"][1:]
        assert np.max(np.abs(t - tr) / tr) < 1e-11
        assert np.max(np.abs(whole["unwrapped"] - ora["unwrapped"])) < 1e-8
        for chunk in (1, 64, 97):
            part = _run(run, table, nc, hops, compact, chunk)
            for key in KEYS:
                assert np.array_equal(part[key], whole[key]), (key, chunk)
            assert part["occupancy"] == whole["occupancy"]
            assert part["energy_now"] == whole["energy_now"]


def test_refusals_name_their_limits():
    w = workloads.corundum(4, n_carriers=122)
    table = w.build_table()
    run = w.make_run(table)
    with pytest.raises(_native.NativeError,
                       match=r"n_c=122, z=4: a session takes n_c \(104 z \+ "
                             r"88\) up to 61424"):
        _native.KmcSession(native_problem(run, table))
    w = workloads.corundum(4, n_carriers=121)
    run = w.make_run(table)
    sess = _native.KmcSession(native_problem(run, table))
    assert sess.variant() == "workgroup"
    with pytest.raises(_native.NativeError, match="PYCD_KMC_WAVE is for"):
        sess.set_variant("wave")
    sess.close()
