"""The work that users of this framework have it do, as timed cases.

Two families, through the package's public entry points:

* stochastic simulation of a reaction network (Sim, Batch, SweepProblem):
  the Schlogl model the reference ships, the 100x200 mass-action network of
  the benchmark, the enzyme cascade, the 50x100 network of the parameter
  sweep, uneven batches of models; adaptive tau-leaping and exact SSA; the
  outputs a user reads back (raw samples in either layout, final states,
  moments, fitness values);
* the sweep's surrogate network (MLP): inference, one gradient, training.

A case is a dict of plain values.  `prepare` builds what a program holds
before the call (the compiled model, the simulation handle, the network with
its weights, the input arrays), `run` is one call of the entry points with
their outputs, `work` the bytes and operations the call cannot do without.
Philox seeds, rate rows, initial counts, weights and training rows come from
`prepare`'s seed; a network and its nominal constants belong to the case.
"""
import functools
import os
import tempfile

import numpy as np
import torch

import cutauleaping_amd as ctl
from cutauleaping_amd import networks
from cutauleaping_amd.surrogate import SweepProblem

# Mass-action networks (species, reactions, generator seed): accepted leaps
# and SSA steps of one adaptive simulation up to t = 0.05, 0.5 and 5 (means of
# a few host simulations), for `work` and for bounding what `draw` asks for.
NETS = {
    (13, 29, 1): ((128, 1300), (321, 1600), (582, 2300)),
    (25, 61, 1): ((376, 2262), (378, 4625), (388, 9900)),
    (37, 71, 1): ((307, 1888), (411, 1888), (699, 1888)),
    (50, 100, 1): ((2126, 17900), (2341, 23750), (2341, 58475)),
    (64, 128, 1): ((900, 900), (4600, 925), (17700, 925)),
    (75, 150, 1): ((1350, 22250), (1350, 43475), (1824, 125512)),
    (80, 150, 2): ((3000, 4300), (5600, 4337), (12400, 4650)),
    (100, 200, 1): ((2600, 0), (7162, 34), (12357, 38)),
}
NET_TIMES = (0.05, 0.5, 5.0)

# Surrogate widths: the sweep's own, and small and odd ones.
WIDTHS = {"sweep": (32, 256, 256, 256, 1000), "small": (8, 128, 128, 16), "odd": (7, 65, 129, 33)}


def listed():
    return [
        # The reference's own example at its own size: 64 threads x 16 blocks
        # of the Schlogl model, samples in the reference's layout.
        dict(name="schlogl_1024", kind="schlogl", threads=64, blocks=16, t_end=10.0, K=100, force_ssa=False,
             rows=False, out="samples", layout=0),
        # A parameter scan of a small model: one rate row per simulation, as
        # the reference reads c_matrix, an odd count that fills the chip.
        dict(name="schlogl_scan_50001", kind="schlogl", threads=50001, blocks=1, t_end=2.5, K=25, force_ssa=False,
             rows=True, out="samples", layout=1),
        # Parameter estimation: fitness of candidate rate rows against a
        # target series, every candidate simulated in 8 parallel repetitions.
        dict(name="fitness_512x8", kind="fitness", threads=128, blocks=32, reps=8, t_end=1.0, K=100, targets=2),
        # The smallest calls: a few simulations of the benchmark network.
        dict(name="mass_action_24", kind="mass_action", N=100, M=200, net=1, threads=24, blocks=1, t_end=0.5, K=20,
             observed=10, lanes=0, force_ssa=False, out="samples", layout=1),
        # An ordinary ensemble of the benchmark network, means and deviations.
        dict(name="mass_action_1000", kind="mass_action", N=100, M=200, net=1, threads=40, blocks=25, t_end=5.0, K=50,
             observed=100, lanes=0, force_ssa=False, out="moments", group=500),
        # The benchmark network at the benchmark's horizon, every resident
        # group of the chip busy.
        dict(name="mass_action_16384", kind="mass_action", N=100, M=200, net=1, threads=64, blocks=256, t_end=50.0,
             K=200, observed=100, lanes=0, force_ssa=False, out="moments", group=1024),
        # The enzyme cascade, adaptive (it spends its time in SSA bursts).
        dict(name="cascade_65536", kind="cascade", stages=20, threads=256, blocks=256, t_end=100.0, K=100,
             observed=20, lanes=0, force_ssa=False, out="moments", group=256),
        # Exact SSA of a cascade of another size, an odd number of
        # simulations, raw samples of three species.
        dict(name="cascade_ssa_5003", kind="cascade", stages=13, threads=5003, blocks=1, t_end=50.0, K=50, observed=3,
             lanes=0, force_ssa=True, out="samples", layout=1),
        # A parameter sweep from the problem to its moments: the whole call
        # (model, handle, simulations, moments) as the sweep study makes it.
        dict(name="sweep_128x256", kind="sweep", sets=128, replicas=256, t_end=1.0),
        # An uneven batch of models in one launch sequence.
        dict(name="batch_64", kind="batch", first=0, count=64, replicas=16, t_end=0.001, K=20, force_ssa=False),
        # Surrogate inference on device buffers over a whole sweep's sets.
        dict(name="mlp_forward_65536", kind="mlp_forward", widths="sweep", rows=65536, host=False),
        # One epoch of surrogate training in the study's batches of 256.
        dict(name="mlp_train_8192", kind="mlp_train", widths="sweep", rows=8192, batch=256, epochs=1),
    ]


def _log(rng, lo, hi):
    return lo * (hi / lo) ** rng.random()


def draw(rng):
    kind = rng.choice(["schlogl", "mass_action", "mass_action", "cascade", "cascade", "sweep", "batch", "fitness",
                       "mlp_forward", "mlp_gradient", "mlp_train"])
    if kind == "schlogl":
        return dict(kind=kind, threads=int(_log(rng, 8, 300)), blocks=int(_log(rng, 1, 160)),
                    t_end=round(_log(rng, 0.1, 10.0) if rng.random() < 0.7 else 1.0, 3), K=rng.randint(1, 100),
                    force_ssa=rng.random() < 0.25, rows=rng.random() < 0.5, out="samples", layout=rng.randint(0, 1))
    if kind == "mass_action":
        N, M, net = rng.choice(sorted(NETS))
        threads, blocks = int(_log(rng, 4, 64)), int(_log(rng, 2, 64))
        return dict(kind=kind, N=N, M=M, net=net, threads=threads, blocks=blocks, t_end=round(_log(rng, 0.02, 2.0), 3),
                    K=rng.randint(2, 60), observed=rng.randint(1, N), lanes=rng.choice([0, 0, 0, 8, 16, 32, 64]),
                    force_ssa=False, out=rng.choice(["samples", "moments"]), layout=rng.randint(0, 1), group=threads)
    if kind == "cascade":
        threads, blocks = int(_log(rng, 16, 256)), int(_log(rng, 1, 256))
        stages = rng.randint(3, 40)
        return dict(kind=kind, stages=stages, threads=threads, blocks=blocks, t_end=round(_log(rng, 5.0, 100.0), 2),
                    K=rng.randint(2, 100), observed=rng.randint(1, 3 * stages + 1), lanes=rng.choice([0, 0, 0, 4, 8]),
                    force_ssa=rng.random() < 0.5, out="moments", group=threads)
    if kind == "sweep":
        return dict(kind=kind, sets=int(_log(rng, 1, 120)), replicas=rng.choice([64, 128, 256]),
                    t_end=round(_log(rng, 0.1, 1.0), 3))
    if kind == "batch":
        return dict(kind=kind, first=rng.randint(0, 120), count=int(_log(rng, 3, 64)), replicas=rng.randint(3, 16),
                    t_end=round(_log(rng, 0.0002, 0.001), 6), K=rng.randint(2, 20), force_ssa=False)
    if kind == "fitness":
        reps = rng.choice([1, 2, 4, 8])
        return dict(kind=kind, threads=rng.randint(16, 256), blocks=reps * rng.randint(1, 4), reps=reps,
                    t_end=round(_log(rng, 0.1, 1.0), 3), K=rng.randint(5, 100), targets=rng.randint(1, 3))
    widths = rng.choice(["sweep", "sweep", "small", "odd"])
    if kind == "mlp_forward":
        return dict(kind=kind, widths=widths, rows=int(_log(rng, 1, 60000)), host=rng.random() < 0.3)
    if kind == "mlp_gradient":
        return dict(kind=kind, widths=widths, rows=int(_log(rng, 16, 4096)))
    batch = int(_log(rng, 32, 2048))
    return dict(kind=kind, widths=widths, rows=batch * rng.randint(1, 8) + rng.randint(0, 31), batch=batch,
                epochs=rng.randint(1, 2))


# ---------------------------------------------------------------------------
# Networks
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _mass_action(N, M, net):
    return networks.mass_action(N, M, seed=net, t_end=5.0)


@functools.lru_cache(maxsize=None)
def _sweep(t_end):
    return SweepProblem.synthetic(t_end=t_end)


@functools.lru_cache(maxsize=None)
def _batch_net(i, t_end):
    return networks.batched_model(i, t_end=t_end)


def _network(case):
    if case["kind"] in ("schlogl", "fitness"):
        return networks.schlogl()
    if case["kind"] == "mass_action":
        return _mass_action(case["N"], case["M"], case["net"])
    return networks.enzyme_cascade(case["stages"])


def _observed(case, S):
    if "observed" not in case:
        return None
    return np.sort(np.random.default_rng(S).choice(S, size=min(S, case["observed"]), replace=False)).astype(np.int32)


def _load_targets(model, case, S, ts):
    """Loads fitness inputs, kept as the reference keeps them: text files in a
    folder.  One experiment; `targets` series per sampled species."""
    E = case["targets"]
    level = 100.0 + 400.0 * np.arange(len(ts)) / len(ts)
    table = "".join(f"{t}" + "".join(f"\t100000\t{int(x) + 20 * e}\t200000" for e in range(E)) + "\n"
                    for t, x in zip(ts, level))
    with tempfile.TemporaryDirectory(prefix="targets_") as d:
        for name, text in (("p_rep", f"{case['reps']}\n"), ("ts_rep", f"{E}\n"), ("ts_numtgt", f"{S}\n"),
                           ("tts_vector", f"{case['threads'] * case['blocks']}\n"), ("ts_matrix", table)):
            with open(os.path.join(d, name), "w") as f:
                f.write(text)
        model.load_fitness(d, case["threads"], case["blocks"])


# ---------------------------------------------------------------------------
# Surrogate inputs
# ---------------------------------------------------------------------------
def _mlp_inputs(case, seed):
    """(parameters, x, t) in FP32: He-uniform weights, small biases, inputs in
    the sweep's range, standardised targets."""
    w = WIDTHS[case["widths"]]
    rng = np.random.default_rng([seed, 11])
    params = np.concatenate([v for a, b in zip(w[:-1], w[1:])
                             for v in (rng.uniform(-1, 1, a * b) * np.sqrt(6.0 / a), rng.uniform(-0.1, 0.1, b))])
    x = rng.uniform(-1.0, 1.0, (case["rows"], w[0])).astype(np.float32)
    t = None
    if case["kind"] != "mlp_forward":
        mix = rng.standard_normal((w[0], w[-1])) / np.sqrt(w[0])
        t = (np.tanh(x @ mix) + 0.1 * rng.standard_normal((case["rows"], w[-1]))).astype(np.float32)
    return params.astype(np.float32), x, t


# ---------------------------------------------------------------------------
# prepare / run
# ---------------------------------------------------------------------------
def prepare(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng([seed, 3])
    if kind == "sweep":
        problem = _sweep(case["t_end"])
        return dict(case=case, problem=problem, u=problem.sample_u(case["sets"], rng), seed=seed + 1)
    if kind == "batch":
        nets = [_batch_net(case["first"] + i, case["t_end"]) for i in range(case["count"])]
        ts = networks.sample_times(case["K"], case["t_end"])
        models = [ctl.Model.from_arrays(n["left"], n["right"], n["x0"], n["c"] * rng.uniform(0.9, 1.1, len(n["c"])),
                                        ts, cs=n["cs"]) for n in nets]
        reps = [max(2, n["replicas"] // case["replicas"]) for n in nets]
        return dict(case=case, models=models, batch=ctl.Batch(models, reps, seed=seed + 1,
                                                              force_ssa=case["force_ssa"]))
    if kind.startswith("mlp"):
        params, x, t = _mlp_inputs(case, seed)
        net = ctl.MLP(WIDTHS[case["widths"]], seed=1)
        net.set_params(params)
        s = dict(case=case, net=net, x=x, t=t)
        if kind == "mlp_train":
            net.set_data(x, t)
        elif kind == "mlp_forward" and not case["host"]:
            s["xd"] = torch.from_numpy(x).cuda()
            s["yd"] = torch.empty((case["rows"], WIDTHS[case["widths"]][-1]), dtype=torch.float32, device="cuda")
            torch.cuda.synchronize()
        return s
    net = _network(case)
    R, S = net["left"].shape
    n = case["threads"] * case["blocks"]
    ts = networks.sample_times(case["K"], case["t_end"])
    x0, c, feed = net["x0"], net["c"], net.get("feed")
    if kind == "cascade":
        x0 = np.maximum(0, np.rint(x0 * rng.uniform(0.9, 1.1, S))).astype(np.uint32)
    elif kind == "fitness" or case.get("rows"):
        c = c * 10.0 ** rng.uniform(-0.05, 0.05, (n, R))
    model = ctl.Model.from_arrays(net["left"], net["right"], x0, c, ts, feed=feed, cs=_observed(case, S))
    if kind == "fitness":
        _load_targets(model, case, S, ts)
    sim = ctl.Sim(model, case["threads"], case["blocks"], seed=seed + 1, force_ssa=case.get("force_ssa", False),
                  lanes_per_sim=case.get("lanes", 0))
    return dict(case=case, model=model, sim=sim)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "sweep":
        mean, sd, _, _ = state["problem"].simulate(state["u"], case["replicas"], seed=state["seed"])
        return dict(mean=mean, sd=sd)
    if kind == "batch":
        b = state["batch"].run()
        return np.concatenate([b.samples(i).reshape(-1) for i in range(case["count"])])
    if kind == "mlp_forward":
        if case["host"]:
            return state["net"].forward(state["x"])
        state["net"].forward_device(state["xd"].data_ptr(), case["rows"], state["yd"].data_ptr())
        return state["yd"]
    if kind == "mlp_gradient":
        loss, grad = state["net"].gradient(state["x"], state["t"])
        return dict(loss=loss, grad=grad)
    if kind == "mlp_train":
        losses = state["net"].train(case["epochs"], case["batch"], 1e-3, seed=5)
        return dict(losses=losses, params=state["net"].get_params())
    sim = state["sim"].run()
    if kind == "fitness":
        return sim.fitness(case["blocks"] // case["reps"])
    if case["out"] == "moments":
        mean, sd = sim.moments(case["group"])
        x, t = sim.final_state()
        return dict(mean=mean, sd=sd, x=x, t=t)
    return sim.samples(case["layout"])


# ---------------------------------------------------------------------------
# work / exact
# ---------------------------------------------------------------------------
def _steps(case):
    """(leaps, SSA steps) of one simulation of the case, about."""
    kind, t = case["kind"], case["t_end"]
    if kind in ("schlogl", "fitness"):
        if case.get("force_ssa"):
            return 0.0, 2350.0 * t + 240.0 * t * t
        return 146.0 * t * min(1.0, t / 10.0 + 0.08), 730.0 * t if t > 3 else 2230.0 * t
    if kind == "cascade":
        return 0.03 * t, 40.0 * t
    if kind == "sweep":
        return 950.0 * (t / 0.5) ** 0.4, 62600.0 * (t / 0.5) ** 0.4
    rows = np.array(NETS[(case["N"], case["M"], case["net"])], float)
    lt = np.log(np.clip(t, 0.01, 5.0))
    leaps, ssa = (float(np.interp(lt, np.log(NET_TIMES), rows[:, k])) for k in (0, 1))
    if (case["N"], case["M"]) == (100, 200) and t > 5.0:      # the benchmark's horizon, t = 50
        f = (min(t, 50.0) - 5.0) / 45.0
        leaps, ssa = 12357.0 + f * 19500.0, 38.0 + f * 93000.0
    return leaps, ssa


def _sim_ops(S, R, leaps, ssa):
    """Operations of one simulation: a leap touches every propensity, reactant
    entry, tau' entry and state change of a network of about two reactants and
    two changes per reaction; a direct-method step sums the propensities,
    selects and refreshes the dependent ones."""
    return leaps * (25.0 * R + 8.0 * S) + ssa * (6.0 * R + 40.0 + S)


def work(case):
    kind = case["kind"]
    if kind.startswith("mlp"):
        w, rows = WIDTHS[case["widths"]], case["rows"]
        macs = sum(a * b for a, b in zip(w[:-1], w[1:]))
        params = macs + sum(w[1:])
        if kind == "mlp_forward":
            return {"bytes": 4.0 * (rows * (w[0] + w[-1]) + params), "flops": 2.0 * rows * macs}
        if kind == "mlp_gradient":
            return {"bytes": 4.0 * (rows * (w[0] + w[-1]) + 2 * params), "flops": 6.0 * rows * macs}
        steps = case["epochs"] * (rows // case["batch"])
        return {"bytes": 4.0 * steps * (case["batch"] * (w[0] + w[-1]) + 6 * params),
                "flops": 6.0 * steps * case["batch"] * macs}
    if kind == "batch":
        b = f = 0.0
        for i in range(case["count"]):
            n = _batch_net(case["first"] + i, case["t_end"])
            R, S = n["left"].shape
            reps = max(2, n["replicas"] // case["replicas"])
            b += 4.0 * (R + S + reps * case["K"] * len(n["cs"]))
            f += reps * _sim_ops(S, R, 8.0 * R * (case["t_end"] / 0.02) ** 0.5, 60.0 * R * (case["t_end"] / 0.02) ** 0.5)
        return {"bytes": b, "flops": f}
    if kind == "sweep":
        n = case["sets"] * case["replicas"]
        return {"bytes": 4.0 * (case["sets"] * 100 + 50) + 16.0 * case["sets"] * 500,
                "flops": n * _sim_ops(50, 100, *_steps(case))}
    net = _network(case)
    R, S = net["left"].shape
    n = case["threads"] * case["blocks"]
    SS = min(S, case.get("observed", S))
    rows = n if kind == "fitness" or case.get("rows") else 1
    read = 4.0 * (rows * R + S)
    if kind == "fitness":
        written = 8.0 * n / case["reps"]
    elif case["out"] == "moments":
        written = 16.0 * (n // case["group"]) * case["K"] * SS + n * (4.0 * S + 8.0)
    else:
        written = 4.0 * n * case["K"] * SS
    return {"bytes": read + written, "flops": n * _sim_ops(S, R, *_steps(case))}


def exact(case, seed):
    """The surrogate's outputs in 64 bits.  A simulation's outputs are whole
    numbers of its random streams, or averages of them: they have no other
    value than the framework's own.  Training is left out: its batches come
    from the library's own shuffle."""
    if case["kind"] not in ("mlp_forward", "mlp_gradient"):
        return None
    w = WIDTHS[case["widths"]]
    params, x, t = _mlp_inputs(case, seed)
    p, acts, layers, o = params.astype(np.float64), [x.astype(np.float64)], [], 0
    for a, b in zip(w[:-1], w[1:]):
        W, o = p[o:o + a * b].reshape(a, b), o + a * b
        bias, o = p[o:o + b], o + b
        layers.append(W)
        z = acts[-1] @ W + bias
        acts.append(np.maximum(z, 0.0) if len(layers) < len(w) - 1 else z)
    if case["kind"] == "mlp_forward":
        return torch.from_numpy(acts[-1]) if not case["host"] else acts[-1]
    e = acts[-1] - t.astype(np.float64)
    loss = float(np.mean(e * e))
    e = 2.0 * e / e.size
    parts = []
    for k in range(len(layers) - 1, -1, -1):
        parts.append(np.concatenate([(acts[k].T @ e).reshape(-1), e.sum(axis=0)]))
        if k:
            e = (e @ layers[k].T) * (acts[k] > 0.0)
    return dict(loss=loss, grad=np.concatenate(parts[::-1]))
