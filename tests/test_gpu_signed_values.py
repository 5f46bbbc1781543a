"""Inputs that make propensities negative -- negative rate constants, counts of 2^31 and more -- run on the kernels
that keep their sign, whatever the library would pick by size: the default geometry gives what an explicit one
gives, and every run ends."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LEFT = [[3, 0, 0, 0], [0, 2, 0, 0], [1, 1, 0, 0], [0, 0, 1, 0], [0, 0, 0, 1], [1, 0, 0, 0], [0, 1, 1, 0]]
RIGHT = [[0, 0, 1, 0], [0, 0, 1, 0], [0, 0, 0, 1], [1, 0, 0, 0], [0, 1, 0, 0], [0, 1, 0, 0], [0, 0, 0, 2]]
RATES = np.array([1e-5, 1e-3, 1e-3, 0.5, 0.4, 0.3, 1e-3])
SCALE = np.array([1e-4, 1e-2, 1e-2, 1, 1, 1, 1e-2])             # the same rates per molecule at 100 times the counts
X0 = np.array([[300, 200, 150, 100]], np.uint32)
BIG = 2**31 + 7


def _inputs(kind, large):
    x0, c = (X0 * 100, RATES * SCALE) if large else (X0.copy(), RATES.copy())
    if kind == "rate":
        c[3] = -c[3]
    else:
        c[4] = 2e-8
        if kind == "count":
            x0[0, 3] = BIG
    return x0, c


@pytest.mark.parametrize("order", [3, 2])
@pytest.mark.parametrize("kind,large", [("rate", False), ("rate", True), ("count", False), ("count", True),
                                        ("feed", True)])
@pytest.mark.parametrize("lanes,explicit", [(1, {"block_size": 64}), (4, {"slots": 40}), (16, {"slots": 40})])
@pytest.mark.parametrize("force", [False, True])
def test_default_geometry_equals_explicit(gpu, order, kind, large, lanes, explicit, force):
    print(f"case: signed {kind} large={large} order={order} lanes={lanes} force={force}", flush=True)
    left = [[order, 0, 0, 0]] + LEFT[1:]
    x0, c = _inputs(kind, large)
    m = gpu.Model.from_arrays(left, RIGHT, x0, [c], np.linspace(0.02, 0.2, 6) if large else np.linspace(0.2, 2.0, 6))
    if kind == "feed":
        m.set_feeds([3], np.array([[BIG]], np.uint32))
    got = []
    for geom in ({}, explicit):
        with gpu.Sim(m, 40, 1, seed=3, lanes_per_sim=lanes, force_ssa=force, **geom) as s:
            s.run()
            got.append((s.samples(), s.sim_stats(), *s.final_state()))
    m.close()
    a, b = got
    for f in a[1].dtype.names:
        assert np.array_equal(a[1][f], b[1][f], equal_nan=f == "t_end"), f
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[2], b[2]) and np.array_equal(a[3], b[3], equal_nan=True)


def test_batch_with_a_negative_rate(gpu):
    print("case: signed batch", flush=True)
    got = []
    for geom in ({}, {"slots": 200}):
        ms = [gpu.Model.from_arrays(LEFT, RIGHT, *_inputs(k, large), np.linspace(0.02, 0.2, 6))
              for k, large in (("rate", True), ("count", False), ("none", True))]
        with gpu.Batch(ms, [40, 40, 40], seed=3, lanes_per_sim=4, **geom) as b:
            b.run()
            got.append([b.samples(i) for i in range(3)])
        for m in ms:
            m.close()
    assert all(np.array_equal(u, v) for u, v in zip(*got))
