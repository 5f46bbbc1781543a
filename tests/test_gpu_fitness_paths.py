"""The fitness values by a thread and by a wavefront each, at the edges of the rule between them, against the same
arithmetic in numpy (sums of integers, IEEE divisions and an FP32 chain: equal to the last bit)."""
import numpy as np
import pytest

from cutauleaping_amd.networks import sample_times, schlogl

pytestmark = pytest.mark.gpu


# 16 loads a value and 8192 values; one repetition and 65536 to 262144 values
@pytest.mark.parametrize("K,cs,E,P,threads,blocks", [
    (8, [0, 1], 2, 1, 8191, 1), (8, [0, 1], 2, 1, 4096, 2), (2, [0, 1], 1, 4, 1025, 32), (17, [1], 1, 1, 8192, 1),
    (20, [0, 1, 2], 1, 1, 65535, 1), (20, [0, 1, 2], 3, 1, 16384, 4), (7, [0, 1, 2], 1, 1, 65535, 4),
    (7, [0, 1, 2], 2, 1, 52430, 5), (7, [0, 1, 2], 1, 2, 65536, 2),
])
def test_fitness_by_size_equals_reference_arithmetic(gpu, tmp_path, K, cs, E, P, threads, blocks):
    print(f"case: fitness K={K} cs={cs} E={E} P={P} {threads}x{blocks}", flush=True)
    net, n, SS, D, groups = schlogl(), threads * blocks, len(cs), 2, blocks // P
    rng = np.random.default_rng(K + threads)
    tgt = rng.integers(0, 600, (K, D, E, SS))
    tgt[rng.random(tgt.shape) < 0.2] = 0
    for name, text in (("p_rep", f"{P}\n"), ("ts_rep", f"{E}\n"), ("ts_numtgt", f"{SS}\n"),
                       ("tts_vector", f"{n // 3}\n{n}\n"),
                       ("ts_matrix", "".join("\t".join(["0"] + [str(v) for v in r]) + "\n" for r in tgt.reshape(K, -1)))):
        (tmp_path / name).write_text(text)
    m = gpu.Model.from_arrays(net["left"], net["right"], net["x0"], net["c"], sample_times(K, 0.01), feed=net["feed"],
                              cs=cs)
    m.load_fitness(str(tmp_path), threads, blocks)
    with gpu.Sim(m, threads, blocks, seed=9) as s:
        s.run()
        out, fit = s.samples().reshape(groups, P, threads, K, SS), s.fitness(groups)
    m.close()
    mean = out.astype(np.float64).sum(axis=1).reshape(groups * threads, K, SS) / P
    experiment = (np.arange(groups * threads) >= n // 3).astype(int)
    sub = np.zeros(groups * threads, np.float32)
    for k in range(K):
        for q in range(SS):
            for e in range(E):
                t = tgt[k, experiment, e, q].astype(np.float64)
                d = np.abs(t - mean[:, k, q])
                d = np.where(t != 0, d / np.where(t != 0, t, 1.0), d)
                sub = (sub.astype(np.float64) + d).astype(np.float32)
    assert np.array_equal(fit, (1.0 / K) * (1.0 / SS) * sub.astype(np.float64))
