"""The one-lane kernel of small models (tables and reactant factors in LDS)
against the oracle: samples, counters and final states bit-exact."""
import numpy as np
import pytest

from test_gpu_parity import _compare, _random_case

pytestmark = pytest.mark.gpu


# reactions around the batches of 4 and 8; n around the lane layouts (one
# simulation per wavefront up to 4096, two up to 8192, else 64)
@pytest.mark.parametrize("N,M,n,per_sim,kw", [
    (2, 1, 1, False, {}),
    (3, 4, 65, True, {"iters_per_launch": 3}),
    (6, 5, 200, True, {"ssa_chunk": 7, "iters_per_launch": 11}),
    (8, 8, 33, False, {}),
    (9, 9, 70, True, {"force_ssa": True, "iters_per_launch": 2, "ssa_steps": 13}),
    (17, 24, 40, False, {"nc": 0}),
    (12, 31, 129, False, {"nc": 1, "slots": 64}),
    (4, 7, 4097, False, {}),
    (4, 7, 8193, False, {}),
    (31, 1, 10, False, {}),
])
def test_small_networks_bit_exact(gpu, oracle_lib, N, M, n, per_sim, kw):
    print(f"case: small N={N} M={M} n={n} {kw}", flush=True)
    net, feed, x0, c, cs, ts = _random_case(500 + M, N, M, n, per_sim)
    x0 = np.minimum(x0, 4000).astype(np.uint32)
    ts = ts * 0.1
    m = gpu.Model.from_arrays(net["left"], net["right"], x0, c, ts, feed=feed, cs=cs)
    with gpu.Sim(m, n, 1, seed=n + M, offset=5, lanes_per_sim=1, **kw) as s:
        s.run()
        ok = {k: v for k, v in kw.items() if k in ("force_ssa", "nc", "ssa_steps")}
        out, st, xf = oracle_lib.run(net["left"], net["right"], x0, c, ts, locked=feed, cs=cs, n=n, seed=n + M,
                                     sim_base=5, final=True, **ok)
        _compare(s, out, st, xf)
    m.close()


@pytest.mark.parametrize("force", [False, True])
def test_small_orders_and_counts_bit_exact(gpu, oracle_lib, force):
    """Multiplicities 1 to 3, alone and with a second reactant, from counts 0 to 4 up; a reaction that changes
    nothing, one without dependents, one without reactants."""
    left = [[3, 0, 0, 0], [2, 1, 0, 0], [1, 1, 0, 0], [0, 0, 0, 0], [1, 0, 0, 0], [0, 3, 1, 0], [0, 0, 1, 0]]
    right = [[2, 0, 0, 0], [2, 0, 0, 1], [0, 1, 1, 0], [0, 1, 0, 0], [1, 0, 0, 0], [1, 2, 0, 0], [0, 0, 0, 1]]
    x0 = np.array([[a, b, c, 0] for a in (0, 1, 2, 3, 4, 40) for b in (0, 1, 2, 3, 300) for c in (0, 1, 50)],
                  np.uint32)
    c = [[0.02, 0.01, 0.05, 3.0, 0.3, 0.02, 0.4]]
    ts = np.linspace(0.1, 4.0, 23)
    m = gpu.Model.from_arrays(left, right, x0, c, ts)
    with gpu.Sim(m, len(x0), 1, seed=3, force_ssa=force, lanes_per_sim=1) as s:
        s.run()
        out, st, xf = oracle_lib.run(left, right, x0, c, ts, n=len(x0), seed=3, force_ssa=force, final=True)
        _compare(s, out, st, xf)
    m.close()
