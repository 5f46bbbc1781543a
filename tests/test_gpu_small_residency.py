"""Which kernel and how many lanes of a wavefront a small model's run gets: the run has to be resident as a whole where
one of the kernels can hold it, and every choice computes the same simulations."""
import numpy as np
import pytest

from test_gpu_parity import _compare

pytestmark = pytest.mark.gpu


def _closed(S, R, order, x):
    """R reactions of up to `order` molecules that keep the number of molecules; the first takes `order` of one kind."""
    rng = np.random.default_rng([S, R, order])
    left, right, c = np.zeros((R, S), int), np.zeros((R, S), int), np.zeros((1, R))
    for j in range(R):
        k = order if j == 0 else int(rng.integers(1, min(order, S) + 1))
        for s in [0] * k if j == 0 else rng.choice(S, k, replace=False):
            left[j, s] += 1
        right[j] = left[j]
        while np.array_equal(right[j], left[j]):
            right[j] = np.bincount(rng.integers(0, S, k), minlength=S)
        c[0, j] = rng.uniform(0.5, 2.0) * x ** (1.0 - k)
    return left, right, rng.integers(x // 2, 2 * x, (1, S)).astype(np.uint32), c


def _check(gpu, oracle_lib, S, R, order, n, x, t, resident, **kw):
    print(f"case: small residency S={S} R={R} order={order} n={n} x={x} {kw}", flush=True)
    left, right, x0, c = _closed(S, R, order, x)
    ts = np.array([t / 2, t])
    m = gpu.Model.from_arrays(left, right, x0, c, ts)
    with gpu.Sim(m, n, 1, seed=n, lanes_per_sim=1, **kw) as s:
        s.run()
        assert not resident or s.stats()["slots"] >= n
        _compare(s, *oracle_lib.run(left, right, x0, c, ts, n=n, seed=n, final=True, threads=8,
                                    force_ssa=kw.get("force_ssa", False)))
    m.close()


# the table of 2 species and 58 reactions leaves 10 wavefronts a CU, not 16: 4096 simulations go two to a wavefront;
# 64 simulations of the others fill an LDS of three or six wavefronts, tau_leap_kernel holds nine
@pytest.mark.parametrize("S,R,order,n", [(2, 58, 2, 4096), (20, 20, 3, 50001), (28, 6, 3, 50001), (16, 30, 2, 110003)])
def test_a_run_that_fits_is_resident(gpu, oracle_lib, S, R, order, n):
    _check(gpu, oracle_lib, S, R, order, n, 400, 0.02, True)


# the lane rules' edges: 1 / 2 / 64 lanes, and with more than two species per reaction 1 / 2 / 4 / 64
@pytest.mark.parametrize("S,R,order,n", [
    (9, 6, 2, 4097), (2, 58, 2, 2561), (13, 6, 2, 512), (13, 6, 2, 513), (13, 6, 2, 1025), (13, 6, 2, 1665),
    (13, 6, 2, 3073), (13, 6, 2, 6145), (13, 6, 2, 8191), (13, 6, 2, 12289), (13, 6, 3, 512), (13, 6, 3, 513),
])
def test_lane_layouts_bit_exact(gpu, oracle_lib, S, R, order, n):
    _check(gpu, oracle_lib, S, R, order, n, 300, 0.1, True)


# beyond the residency: force-SSA runs stay, or move where there are few reactions to a simulation's words
@pytest.mark.parametrize("S,R,order,n,kw", [
    (16, 30, 2, 110003, {"force_ssa": True}), (30, 4, 2, 90001, {"force_ssa": True}),
    (8, 24, 2, 200003, {}), (8, 24, 2, 270001, {}), (16, 30, 2, 900, {"slots": 192}),
    (28, 6, 3, 400, {"slots": 64, "iters_per_launch": 5}),
])
def test_beyond_the_residency_bit_exact(gpu, oracle_lib, S, R, order, n, kw):
    _check(gpu, oracle_lib, S, R, order, n, 60, 0.05, False, **kw)
