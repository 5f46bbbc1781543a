"""The fitness values against the same arithmetic in numpy (sums of integers,
IEEE divisions and an FP32 chain: equal to the last bit)."""
import numpy as np
import pytest

from cutauleaping_amd.networks import sample_times, schlogl

pytestmark = pytest.mark.gpu


# K * species * repetitions around the 64 distances of a pass: 1, 60, 63, 64, 66, 130
@pytest.mark.parametrize("K,cs,E,D,P,threads,blocks", [
    (1, [1], 1, 1, 1, 1, 1),
    (20, [0, 1, 2], 1, 2, 3, 5, 9),
    (7, [0, 1, 2], 3, 1, 1, 33, 2),
    (32, [1], 2, 3, 8, 7, 16),
    (33, [1, 2], 1, 2, 4, 64, 7),
    (13, [1, 2], 5, 4, 2, 16, 6),
])
def test_fitness_equals_reference_arithmetic(gpu, tmp_path, K, cs, E, D, P, threads, blocks):
    print(f"case: fitness K={K} cs={cs} E={E} D={D} P={P} {threads}x{blocks}", flush=True)
    net, n, SS = schlogl(), threads * blocks, len(cs)
    rng = np.random.default_rng(K * 100 + E)
    tgt = rng.integers(0, 600, size=(K, D * E * SS))
    tgt[rng.random(tgt.shape) < 0.2] = 0
    ends = np.sort(rng.integers(0, n + 1, size=D))
    ends[-1] = n
    (tmp_path / "p_rep").write_text(f"{P}\n")
    (tmp_path / "ts_rep").write_text(f"{E}\n")
    (tmp_path / "ts_numtgt").write_text(f"{SS}\n")
    (tmp_path / "tts_vector").write_text("".join(f"{e}\n" for e in ends))
    (tmp_path / "ts_matrix").write_text("".join("\t".join(["0"] + [str(v) for v in r]) + "\n" for r in tgt))
    m = gpu.Model.from_arrays(net["left"], net["right"], net["x0"], net["c"], sample_times(K, 0.3), feed=net["feed"],
                              cs=cs)
    m.load_fitness(str(tmp_path), threads, blocks)
    groups = blocks // P
    with gpu.Sim(m, threads, blocks, seed=9) as s:
        s.run()
        out, fit = s.samples().reshape(blocks, threads, K, SS), s.fitness(groups)
    exp_of = np.zeros(n, int)
    last = 0
    for d, e in enumerate(ends):
        exp_of[last:e] = d
        last = e
    ref = np.zeros(threads * groups)
    for tid in range(threads * groups):
        g, th = divmod(tid, threads)
        sub = np.float32(0)
        for i in range(K):
            for k in range(SS):
                acc = float(out[g * P:(g + 1) * P, th, i, k].astype(np.int64).sum()) / P
                for r in range(E):
                    t = float(tgt[i, exp_of[tid] * SS * E + r * SS + k])
                    d = abs(t - acc)
                    sub = np.float32(float(sub) + (d / t if t else d))
        ref[tid] = (1.0 / K) * (1.0 / SS) * float(sub)
    assert np.array_equal(fit, ref)
    m.close()
