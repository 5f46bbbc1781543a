"""Counts at the top of their range, against the oracle: leaps rejected because a species would pass 2^31 - 1, on the
update's 32-bit sums and on its 64-bit ones, and leaps with more firings than the 32-bit sums may hold."""
import numpy as np
import pytest

from test_gpu_parity import _compare

pytestmark = pytest.mark.gpu

TOP = 2**31 - 1
# B <-> C, B makes A: A climbs to the top of its range; s molecules of A at a time
UP = lambda s: ([[0, 1, 0], [0, 0, 1], [0, 1, 0]], [[0, 0, 1], [0, 1, 0], [s, 1, 0]])


# 1000 of B and C: leaps of a few hundred firings (32-bit sums); 2e8: leaps of millions (64-bit sums)
@pytest.mark.parametrize("G,n,geom", [(2, 9, {}), (4, 9, {}), (16, 9, {"slots": 9}), (64, 5, {}), (8, 40, {"slots": 16})])
@pytest.mark.parametrize("s,below,bc,c,t", [
    (1, 1500, 1000, (1.0, 1.0, 1.0), 1.6),
    (3, 1500, 1000, (1.0, 1.0, 0.4), 1.4),
    (1, 40_000_000, 200_000_000, (1.0, 1.0, 1e-1), 1.9995),
    (700, 900_000_000, 200_000_000, (1.0, 1.0, 1e-2), 0.6432),
])
def test_leaps_past_the_top_are_rejected(gpu, oracle_lib, G, n, geom, s, below, bc, c, t):
    print(f"case: top G={G} n={n} {geom} step={s} below={below}", flush=True)
    left, right = UP(s)
    x0, ts = np.array([[TOP - below, bc, bc]], np.uint32), np.linspace(t / 7, t, 7)
    out, st, xf = oracle_lib.run(left, right, x0, [c], ts, n=n, seed=3, final=True, group=G)
    assert st["rejections"].sum() > n and st["leaps"].min() > 3 and xf[:, 0].max() > TOP - 4000
    m = gpu.Model.from_arrays(left, right, x0, [c], ts)
    with gpu.Sim(m, n, 1, seed=3, lanes_per_sim=G, **geom) as sim:
        sim.run()
        _compare(sim, out, st, xf)
    m.close()


@pytest.mark.parametrize("G,n,geom", [(4, 9, {}), (16, 9, {"slots": 9}), (16, 2, {}), (64, 5, {})])
def test_firings_beyond_the_32_bit_sums(gpu, oracle_lib, G, n, geom):
    print(f"case: many firings G={G} n={n} {geom}", flush=True)
    rng = np.random.default_rng(8)
    S, R = 20, 40
    left, right = np.zeros((R, S), int), np.zeros((R, S), int)
    for j in range(R):
        a, b = rng.choice(S, 2, replace=False)
        left[j, a], right[j, b] = 1, 1
    x0, ts = rng.integers(20_000_000, 90_000_000, (1, S)).astype(np.uint32), np.linspace(0.3, 3.0, 5)
    c = rng.uniform(0.5, 2.0, (1, R))
    out, st, xf = oracle_lib.run(left, right, x0, c, ts, n=n, seed=5, final=True, group=G)
    assert (st["firings"] / st["leaps"]).min() > 2**23          # the 32-bit sums' bound over all lanes
    m = gpu.Model.from_arrays(left, right, x0, c, ts)
    with gpu.Sim(m, n, 1, seed=5, lanes_per_sim=G, **geom) as sim:
        sim.run()
        _compare(sim, out, st, xf)
    m.close()


@pytest.mark.parametrize("G,geom", [(2, {"slots": 12}), (4, {"slots": 12}), (16, {}), (64, {}), (8, {"compact_interval": 2})])
def test_runs_with_a_count_above_the_top_end(gpu, oracle_lib, G, geom):
    """A count of 2^31 or more runs as a negative one: no leap can be accepted (a species below 0 rejects whatever is
    drawn), so every attempt has to give up for an SSA burst."""
    print(f"case: above the top G={G} {geom}", flush=True)
    left, right = [[1, 0, 0], [0, 1, 0], [1, 0, 0]], [[0, 1, 0], [1, 0, 0], [1, 0, 1]]
    c, ts = [[1.0, 1.0, 1e-6]], np.array([0.5, 1.0])
    x0 = np.array([[3000, 3000, 2**31 + 7], [3000, 3000, 10]], np.uint32)
    out, st, xf = oracle_lib.run(left, right, x0.repeat(6, axis=0), c, ts, n=12, seed=1, final=True, group=G)
    assert st["leaps"][:6].max() == 0 and st["rejections"][:6].min() > 100 and st["leaps"][6:].min() > 0
    m = gpu.Model.from_arrays(left, right, x0.repeat(6, axis=0), c, ts)
    with gpu.Sim(m, 12, 1, seed=1, lanes_per_sim=G, **geom) as sim:
        sim.run()
        _compare(sim, out, st, xf)
    m.close()
    models = [gpu.Model.from_arrays(left, right, x, c, ts) for x in x0]
    with gpu.Batch(models, [6, 6], seed=1, lanes_per_sim=G) as b:
        b.run()
        for i in range(2):
            assert np.array_equal(b.samples(i), out[6 * i:6 * i + 6])
    for m in models:
        m.close()
