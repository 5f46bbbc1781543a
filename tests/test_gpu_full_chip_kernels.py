"""The kernels that full chips run -- several simulations per wavefront, as many lanes each as the algorithm has, and the
batch's 32-lane teams -- against the oracle.  Small runs get one wavefront per simulation, so an explicit geometry or
the number of replicas selects them here, and the slot count shows that it did."""
import numpy as np
import pytest

from test_gpu_parity import _compare, _random_case

pytestmark = pytest.mark.gpu

FIELDS = ("firings", "leaps", "rejections", "switches", "ssa_steps", "poisson", "gaps", "events")


def _batch_equals_oracle(gpu, oracle_lib, b, nets, reps, G, seed, offset, **kw):
    for i, (net, ts, cs) in enumerate(nets):
        assert b.model_lanes(i) == G
        out, st = oracle_lib.run(net["left"], net["right"], net["x0"], net["c"], ts, cs=cs, n=reps[i], seed=seed,
                                 sim_base=offset + b.stream_base(i), group=G, **kw)
        assert np.array_equal(b.samples(i), out), i
        gs = b.sim_stats(i)
        for f in FIELDS:
            assert np.array_equal(gs[f].astype(np.int64), st[f].astype(np.int64)), (i, f)


def _nets(gpu, seed, count, most, x_max, horizon=0.5):
    from cutauleaping_amd import networks
    rng = np.random.default_rng(seed)
    nets, models = [], []
    for i in range(count):
        N, M = int(rng.integers(3, most[0])), int(rng.integers(4, most[1]))
        net = networks.mass_action(N, M, seed=300 + i, t_end=0.5, check=False)
        net["x0"] = np.minimum(net["x0"], x_max).astype(np.uint32)
        ts = np.linspace(0.02, 1.0, int(rng.integers(5, 30))) * horizon
        cs = np.arange(min(N, 6), dtype=np.int32)
        models.append(gpu.Model.from_arrays(net["left"], net["right"], net["x0"], net["c"], ts, cs=cs))
        nets.append((net, ts, cs))
    return nets, models, rng


# a slot count keeps as many lanes per simulation as the algorithm has: 64 / G groups of a wavefront run replicas of
# one model, gather their SSA bursts and park in the middle of them
@pytest.mark.parametrize("G,iters,slots,force", [
    (2, 41, 65, False), (4, 37, 33, False), (8, 29, 41, False), (16, 23, 21, False), (32, 19, 7, False),
    (4, 5000, 100, False), (32, 5000, 11, False), (4, 3, 17, True), (16, 2, 9, True),
])
def test_class_kernel_of_g_lanes_bit_exact(gpu, oracle_lib, G, iters, slots, force):
    print(f"case: class kernel G=W={G} iters={iters} slots={slots} force={force}", flush=True)
    nets, models, rng = _nets(gpu, 17 + G, 7, (61, 151), *((300, 0.05) if force else (3000, 0.5)))
    reps = [int(rng.integers(1, 70)) for _ in nets]
    with gpu.Batch(models, reps, seed=771, offset=2, iters_per_launch=iters, lanes_per_sim=G, slots=slots,
                   force_ssa=force) as b:
        for _ in range(2):                               # a second run starts from cleared counters
            b.run()
            st = b.stats()
            per = 64 // G
            assert st["lanes_per_sim"] == G and st["slots"] == min(-(-slots // per), -(-sum(reps) // per)) * per
            assert st["launches"] >= (2 if iters < 100 else 1)
        _batch_equals_oracle(gpu, oracle_lib, b, nets, reps, G, 771, 2, force_ssa=force)
    for m in models:
        m.close()


# more replicas than 64-lane teams have places, fewer than 32-lane ones: two simulations per wavefront
@pytest.mark.parametrize("G,iters", [(2, 0), (4, 30), (8, 0), (16, 25)])
def test_class_kernel_of_32_lanes_bit_exact(gpu, oracle_lib, G, iters):
    print(f"case: class kernel G={G} W=32 iters={iters}", flush=True)
    nets, models, _ = _nets(gpu, 5 + G, 3, (9, 24), 3000)
    reps = [1501, 900, 1200]                             # 3601: W = 64 would need 3601 places of at most 3072
    with gpu.Batch(models, reps, seed=772, lanes_per_sim=G, iters_per_launch=iters) as b:
        b.run()
        assert b.stats()["slots"] == 3602
        _batch_equals_oracle(gpu, oracle_lib, b, nets, reps, G, 772, 0)
    for m in models:
        m.close()


# block_size or slots keep W = G; without a regrouping interval a wavefront's groups gather their bursts
@pytest.mark.parametrize("G,N,M,n,geom", [
    (2, 14, 30, 131, {"block_size": 64}),
    (4, 14, 30, 300, {"block_size": 64}),
    (4, 9, 14, 75, {"block_size": 256, "iters_per_launch": 11}),
    (4, 21, 70, 200, {"slots": 40, "iters_per_launch": 9}),
    (8, 14, 30, 200, {"block_size": 256}),
    (8, 40, 90, 60, {"slots": 24, "iters_per_launch": 13, "force_ssa": True}),
    (16, 14, 30, 200, {"block_size": 128}),
    (16, 60, 130, 40, {"slots": 12, "iters_per_launch": 7}),
    (32, 14, 30, 90, {"block_size": 256, "iters_per_launch": 17}),
    (32, 70, 129, 40, {"slots": 6}),
])
def test_group_kernel_of_g_lanes_bit_exact(gpu, oracle_lib, G, N, M, n, geom):
    print(f"case: group kernel G=W={G} N={N} M={M} n={n} {geom}", flush=True)
    net, feed, x0, c, cs, ts = _random_case(700 + M, N, M, n, True)
    x0 = np.minimum(x0, 4000).astype(np.uint32)
    ts = ts * 0.1
    m = gpu.Model.from_arrays(net["left"], net["right"], x0, c, ts, feed=feed, cs=cs)
    with gpu.Sim(m, n, 1, seed=n + G, offset=9, lanes_per_sim=G, **geom) as s:
        s.run()
        st = s.stats()
        per = st["block_size"] // G                      # simulations of a workgroup at W = G
        assert st["slots"] == -(-min(n, geom.get("slots", n)) // per) * per * G
        out, ost, xf = oracle_lib.run(net["left"], net["right"], x0, c, ts, locked=feed, cs=cs, n=n, seed=n + G,
                                      sim_base=9, force_ssa=geom.get("force_ssa", False), final=True, group=G)
        _compare(s, out, ost, xf)
    m.close()
