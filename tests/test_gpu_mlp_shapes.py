"""The surrogate's products at the edges of their tiles and rules, against the numpy oracle: rows and widths around
32, 64 and 128, inner widths above 256 and more than eight layers (layer by layer instead of one fused pass), batches
that split the weight gradient's k loop, and a smaller batch after a larger one in the same buffers.  Tolerances are
those of test_gpu_mlp (a hidden activation on a BF16 rounding boundary may round the other way)."""
import numpy as np
import pytest

from oracle import mlp as om
from test_gpu_mlp import FWD_REL, GRAD_COS, GRAD_REL, _blocks, _init

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("widths,rows", [
    ([1, 1], 1),
    ([31, 33, 32], 31),
    ([33, 64, 65, 63], 33),
    ([64, 256, 255, 1], 64),
    ([20, 257, 40], 129),
    ([5, 512, 320, 130], 2049),
    ([6, 16, 16, 16, 16, 16, 16, 16, 16, 16, 7], 70),
    ([32, 256, 256, 1000], 4100),
])
def test_edges_match_oracle(ctl, gpu, widths, rows):
    print(f"case: mlp {widths} rows={rows}", flush=True)
    net, p = _init(ctl, widths, seed=rows)
    rng = np.random.default_rng(rows)
    x = rng.uniform(-1, 1, (rows, widths[0])).astype(np.float32)
    t = rng.standard_normal((rows, widths[-1])).astype(np.float32)
    for n in (rows, max(1, rows // 3)):
        y, want = net.forward(x[:n]), om.forward(p, widths, x[:n], bf16=True)
        assert np.all(np.isfinite(y)) and np.linalg.norm(y - want) <= FWD_REL * np.linalg.norm(want)
        loss, g = net.gradient(x[:n], t[:n])
        lw, gw = om.gradient(p, widths, x[:n], t[:n], bf16=True)
        assert loss == pytest.approx(lw, rel=1e-2)
        for lo, hi in _blocks(widths):
            a, b = g[lo:hi].astype(np.float64), gw[lo:hi]
            nb = np.linalg.norm(b)
            if nb == 0:
                assert not a.any()
                continue
            assert np.linalg.norm(a - b) / nb < GRAD_REL
            assert float(a @ b / (np.linalg.norm(a) * nb)) > GRAD_COS
    net.close()
