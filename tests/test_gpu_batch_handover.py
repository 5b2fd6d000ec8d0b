"""Hand-over of trajectories whose paths fill after a few hops."""
import numpy as np
import pytest

from pycd_amd import batch as B, rng
from tests.test_gpu_batch_hop import _lattice

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hops,interval", [(2000, 5e5), (2000, 1e30),
                                           (100, 1e30)])
def test_launches_of_short_trajectories(hops, interval):
    """4096 trajectories that end after about 2 hops (paths full) or after
    their hops, all resident at once, so that wavefronts wait and hand over
    from the first hops on: the same results as without hand-over, in every
    launch, and no more hand-overs than trajectories."""
    fam, _ = _lattice(4, 4)
    n, nc = 4096, 2
    counts = [nc] * n
    occs, words = rng.seeded_starts(5, n, [fam.hop_sites] * n, counts)
    trajs = [dict(family=0, n_carriers=nc, carrier_q=-1.0,
                  field=np.array([1e-6, -2e-6, 5e-7]), kT=1.2e-3,
                  time_interval=interval, ewald_neut=0.0, n_path=401,
                  max_hops=hops) for _ in counts]
    bt = B.KmcBatch([fam], "f64", "f32")
    bt.setup(trajs, occs, words, waves_per_cu=16)
    bt.set_handover(False)
    bt.run()
    ref = bt.results()
    assert bt.handovers() == 0
    bt.set_handover(True)
    for _ in range(3):
        bt.run()
        got = bt.results()
        assert 0 <= bt.handovers() <= n
        for key in ("t", "energy", "hops", "start", "no_select", "done",
                    "drift"):
            assert np.array_equal(got[key], ref[key]), key
    bt.close()
