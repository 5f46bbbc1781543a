"""The totals of the statistics against the per-simulation records."""
import numpy as np
import pytest

from cutauleaping_amd.networks import mass_action, sample_times, schlogl

pytestmark = pytest.mark.gpu

TOTALS = ("firings", "leaps", "rejections", "switches", "ssa_steps", "poisson", "gaps", "absorbed")


@pytest.mark.parametrize("n,lanes", [(1, 1), (255, 16), (257, 1), (40000, 1)])
def test_totals_equal_record_sums(gpu, n, lanes):
    net = schlogl()
    m = gpu.Model.from_arrays(net["left"], net["right"], net["x0"], net["c"], sample_times(3, 0.05), feed=net["feed"])
    with gpu.Sim(m, n, 1, seed=4, lanes_per_sim=lanes) as s:
        for _ in range(2):                               # a second run starts from zero again
            s.run()
            rec, st = s.sim_stats(), s.stats()
            assert {k: st[k] for k in TOTALS} == {k: int(rec[k].astype(np.uint64).sum()) for k in TOTALS
                                                  if k in rec.dtype.names}
    m.close()


def test_batch_totals_equal_record_sums(gpu):
    reps = [1, 300, 64, 257]
    nets = [mass_action(6 + 9 * i, 10 + 40 * i, seed=60 + i, t_end=0.2) for i in range(4)]
    ms = [gpu.Model.from_arrays(d["left"], d["right"], d["x0"], d["c"], sample_times(2, 0.2)) for d in nets]
    with gpu.Batch(ms, reps, seed=3) as b:
        for _ in range(2):
            b.run()
            st = b.stats()
            for k in TOTALS:
                assert st[k] == sum(int(b.sim_stats(i)[k].astype(np.uint64).sum()) for i in range(4)), k
    for m in ms:
        m.close()
