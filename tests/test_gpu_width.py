"""The group kernel with more lanes per simulation than its algorithm has
(small runs spread over the chip): every width the library picks, against the
oracle's group algorithm of the same G -- samples, counters and final states
bit-exact."""
import numpy as np
import pytest

from test_gpu_parity import _compare, _random_case

pytestmark = pytest.mark.gpu


# n picks the width: 64 lanes up to 3072 resident simulations, 32 up to 8192,
# 16 up to 16384; N around and above 64 species takes two rounds of species
@pytest.mark.parametrize("G,N,M,n,geom", [
    (2, 9, 14, 1, {}),
    (2, 14, 30, 65, {"iters_per_launch": 7}),
    (4, 65, 64, 33, {"iters_per_launch": 11}),
    (8, 14, 30, 257, {}),
    (16, 130, 260, 24, {"compact_interval": -1}),
    (32, 70, 129, 40, {"iters_per_launch": 30}),
    (4, 5, 9, 4001, {"iters_per_launch": 60}),
    (16, 6, 17, 4001, {}),
    (4, 5, 9, 9001, {}),
    (8, 9, 20, 50, {"force_ssa": True, "iters_per_launch": 3}),
])
def test_wide_execution_bit_exact(gpu, oracle_lib, G, N, M, n, geom):
    print(f"case: width G={G} N={N} M={M} n={n} {geom}", flush=True)
    net, feed, x0, c, cs, ts = _random_case(300 + M, N, M, n, True)
    x0 = np.minimum(x0, 4000).astype(np.uint32)
    ts = ts * 0.1
    m = gpu.Model.from_arrays(net["left"], net["right"], x0, c, ts, feed=feed, cs=cs)
    with gpu.Sim(m, n, 1, seed=n + G, offset=9, lanes_per_sim=G, **geom) as s:
        s.run()
        assert s.stats()["lanes_per_sim"] == G and s.stats()["slots"] >= 2 * G * n
        out, st, xf = oracle_lib.run(net["left"], net["right"], x0, c, ts, locked=feed, cs=cs, n=n, seed=n + G,
                                     sim_base=9, force_ssa=geom.get("force_ssa", False), final=True, group=G)
        _compare(s, out, st, xf)
    m.close()


def test_wide_high_order_absorbing_and_feeds_bit_exact(gpu, oracle_lib):
    """Reactant entries of multiplicity 3 (the general propensity mode), absorption in both modes, and per-simulation
    feeds."""
    left = [[3, 0, 0], [0, 2, 0], [1, 0, 0], [1, 1, 1], [0, 0, 1]]
    right = [[0, 0, 0], [0, 0, 1], [0, 0, 0], [0, 1, 0], [0, 0, 0]]
    x0 = np.array([[60, 40, 0], [5, 3, 2], [5000, 2000, 300], [2, 1, 7]], np.uint32).repeat(64, axis=0)
    c = [[0.01, 0.05, 0.2, 1e-4, 0.1]]
    ts = np.linspace(0.05, 9.0, 60)
    for force, feeds in ((False, False), (True, False), (False, True)):
        print(f"case: width high order force={force} feeds={feeds}", flush=True)
        m = gpu.Model.from_arrays(left, right, x0, c, ts)
        kw = {}
        if feeds:
            fv = np.arange(256, dtype=np.uint32)[:, None] + 3
            m.set_feeds([1], fv)
            kw = dict(feed_species=[1], feed_values=fv)
        with gpu.Sim(m, 256, 1, seed=5, force_ssa=force, lanes_per_sim=2) as s:
            s.run()
            out, st, xf = oracle_lib.run(left, right, x0, c, ts, n=256, seed=5, force_ssa=force, final=True, group=2,
                                         **kw)
            assert feeds or st["absorbed"].sum() > 0
            _compare(s, out, st, xf)
        m.close()
