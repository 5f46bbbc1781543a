"""The slots of a full chip, for each propensity mode's kernel instance: the instances differ in registers, so the number
of resident simulations has to be asked of the one that runs, and each of them holds three wavefronts a SIMD."""
import numpy as np
import pytest

from test_gpu_parity import _compare

pytestmark = pytest.mark.gpu


def _ring(S, R, order):
    """Conversions along a ring of species; the first reaction takes `order` molecules at once."""
    left, right = np.zeros((R, S), int), np.zeros((R, S), int)
    for j in range(R):
        left[j, j % S] = right[j, (j + 1) % S] = 1
    left[0, 0] = right[0, 1] = order
    c = np.full((1, R), 1.0)
    c[0, 0] = 1e-5 if order == 3 else 1.0
    return left, right, c


# three molecules of a species (mode 0), a factor table (1: 2S + 1 <= R + 1 padded to 4), without one (2)
@pytest.mark.parametrize("S,R,order", [(22, 24, 3), (13, 40, 1), (22, 24, 1)])
def test_a_full_chip_holds_three_wavefronts_a_simd(gpu, oracle_lib, S, R, order):
    print(f"case: residency S={S} R={R} order={order}", flush=True)
    left, right, c = _ring(S, R, order)
    x0, ts = np.full((1, S), 30, np.uint32), np.array([0.01, 0.02])
    m = gpu.Model.from_arrays(left, right, x0, c, ts)
    with gpu.Sim(m, 65536, 1, seed=3, lanes_per_sim=4) as s:
        s.run()
        assert s.stats()["slots"] >= 196608              # 256 CUs x 12 wavefronts of 64
        out, _ = oracle_lib.run(left, right, x0, c, ts, n=65536, seed=3, group=4, threads=8)
        assert np.array_equal(s.samples(), out)
    m.close()


@pytest.mark.parametrize("G,S,R,order", [(2, 22, 24, 1), (4, 22, 24, 3), (4, 13, 40, 1), (4, 22, 24, 1)])
def test_regrouping_holds_three_wavefronts_a_simd(gpu, oracle_lib, G, S, R, order):
    print(f"case: residency regrouping G={G} S={S} R={R} order={order}", flush=True)
    left, right, c = _ring(S, R, order)
    x0, ts = np.full((1, S), 30, np.uint32), np.array([0.01, 0.02])
    m = gpu.Model.from_arrays(left, right, x0, c, ts)
    with gpu.Sim(m, 131072, 1, seed=3, lanes_per_sim=G, compact_interval=8) as s:
        s.run()
        assert s.stats()["slots"] >= 196608
        out, _ = oracle_lib.run(left, right, x0, c, ts, n=4096, seed=3, group=G, threads=8)
        assert np.array_equal(s.samples()[:4096], out)
    m.close()


# more simulations than one instance's 64-lane teams hold, fewer than another's
@pytest.mark.parametrize("S,R,order", [(22, 24, 3), (13, 40, 1), (22, 24, 1)])
def test_widths_around_the_residency_bit_exact(gpu, oracle_lib, S, R, order):
    print(f"case: residency widths S={S} R={R} order={order}", flush=True)
    left, right, c = _ring(S, R, order)
    n, x0, ts = 3001, np.full((1, S), 300, np.uint32), np.array([0.05, 0.1])
    m = gpu.Model.from_arrays(left, right, x0, c, ts)
    with gpu.Sim(m, n, 1, seed=3, lanes_per_sim=4) as s:
        s.run()
        _compare(s, *oracle_lib.run(left, right, x0, c, ts, n=n, seed=3, final=True, group=4))
    m.close()


def test_a_batch_of_one_lane_models_has_a_wavefront_per_chunk(gpu, oracle_lib):
    print("case: residency batch", flush=True)
    cases = [_ring(5, 9, 1), _ring(7, 8, 1)]
    x0, ts, reps = [np.full((1, S), 20, np.uint32) for S in (5, 7)], np.array([0.01, 0.02]), [65, 60001]
    ms = [gpu.Model.from_arrays(l, r, x, c, ts) for (l, r, c), x in zip(cases, x0)]
    with gpu.Batch(ms, reps, seed=3) as b:
        b.run()
        assert b.stats()["slots"] == -(-(2 + 938) * 64 // 256) * 256        # chunks of 64, workgroups of 256 lanes
        for i, (l, r, c) in enumerate(cases):
            assert b.model_lanes(i) == 1
            out, _ = oracle_lib.run(l, r, x0[i], c, ts, n=reps[i], seed=3, sim_base=b.stream_base(i), threads=8)
            assert np.array_equal(b.samples(i), out), i
    for m in ms:
        m.close()
