"""Training steps and the 128 x 128 products of the surrogate's network.

The products' tolerances are those of test_gpu_mlp.  A step's: the gradient of a batch differs from the one that
`gradient` returns by the order of its FP32 sum only (training permutes the rows), a relative error of at most
sqrt(rows) 2^-24 < 3e-6 of the gradient's scale for these batches, so below 1e-3 of itself wherever the gradient
is at least 1e-2 of its block's root mean square (in every step so far).  Adam's quotient of moments is homogeneous in
the gradients: there it is off by less than 5e-3 of lr, on top of the FP32 rounding of the parameter."""
import numpy as np
import pytest

from oracle import mlp as om
from test_gpu_mlp import FWD_REL, GRAD_COS, GRAD_REL, _blocks, _init

pytestmark = pytest.mark.gpu


def _data(widths, rows, seed):
    rng = np.random.default_rng(seed)
    return (rng.uniform(-1, 1, (rows, widths[0])).astype(np.float32),
            rng.standard_normal((rows, widths[-1])).astype(np.float32))


# every product of a layer with 256 tiles of 128 x 128 or more: [40, 1000, 1001] x 4200 rows (forward with ReLU, the
# output error, the input error, inference), [30, 2050, 2049, 70] (a weight gradient of 2050 x 2049)
@pytest.mark.parametrize("widths,rows", [([40, 1000, 1001], 4200), ([30, 2050, 2049, 70], 300)])
def test_big_tiles_match_oracle(ctl, gpu, widths, rows):
    print(f"case: mlp big tiles {widths} rows={rows}", flush=True)
    net, p = _init(ctl, widths, seed=rows)
    x, t = _data(widths, rows, rows)
    y, want = net.forward(x), om.forward(p, widths, x, bf16=True)
    assert np.all(np.isfinite(y)) and np.linalg.norm(y - want) <= FWD_REL * np.linalg.norm(want)
    # the last columns and rows, where tiles are cut off, on their own
    assert np.linalg.norm((y - want)[:, -1]) <= FWD_REL * np.linalg.norm(want[:, -1])
    assert np.linalg.norm((y - want)[-1]) <= FWD_REL * np.linalg.norm(want[-1])
    loss, g = net.gradient(x, t)
    lw, gw = om.gradient(p, widths, x, t, bf16=True)
    assert loss == pytest.approx(lw, rel=1e-2)
    for lo, hi in _blocks(widths):
        a, b = g[lo:hi].astype(np.float64), gw[lo:hi]
        nb = np.linalg.norm(b)
        assert nb > 0 and np.linalg.norm(a - b) / nb < GRAD_REL
        assert float(a @ b / (np.linalg.norm(a) * nb)) > GRAD_COS
    net.close()


# ragged widths; more than eight layers (two launches of the fused step); batches above 2048 (separate Adam); a batch
# smaller than the buffers; one tile and one column
@pytest.mark.parametrize("widths,batch,cap", [
    ([7, 65, 129, 33], 97, 0),
    ([32, 256, 256, 256, 1000], 256, 0),
    ([6, 17, 16, 33, 15, 16, 31, 16, 16, 18, 7], 70, 0),
    ([1, 1], 3, 0),
    ([5, 40, 31], 33, 300),
    ([7, 65, 129, 33], 2048, 0),
    ([7, 65, 129, 33], 2049, 0),
    ([9, 2050, 2049, 5], 64, 0),
])
def test_training_steps(ctl, gpu, widths, batch, cap):
    print(f"case: mlp steps {widths} batch={batch} cap={cap}", flush=True)
    net, p = _init(ctl, widths, seed=5)
    x, t = _data(widths, batch, 31 + batch)
    if cap:                                              # buffers (and leading dimensions) of a larger batch first
        net.gradient(*_data(widths, cap, 2))
    net.set_data(x, t)
    lr, b1, b2, eps = (np.float32(v) for v in (1e-2, 0.9, 0.999, 1e-8))
    m, v, firm = np.zeros_like(p), np.zeros_like(p), np.ones(p.size, bool)
    for step in (1, 2):
        _, g = net.gradient(x, t)
        net.train(1, batch, float(lr), seed=step)
        got = net.get_params()
        m = b1 * m + (1 - b1) * g
        v = b2 * v + (1 - b2) * g * g
        c1, c2 = np.float32(1) - b1 ** np.float32(step), np.float32(1) - b2 ** np.float32(step)
        want = p - lr * (m / c1) / (np.sqrt(v / c2) + eps)
        for lo, hi in _blocks(widths):
            gb = np.abs(g[lo:hi])
            firm[lo:hi] &= (gb > 0) & (gb >= 1e-2 * np.sqrt(np.mean(gb.astype(np.float64) ** 2)))
        assert firm.sum() > 0.4 * np.count_nonzero(g)
        d = np.abs(got.astype(np.float64) - want)
        assert np.all(d[firm] <= 5e-3 * lr + 2.0 ** -23 * np.abs(want[firm])), (step, d[firm].max())
        assert np.all(np.abs(got - p) <= 1.1 * lr)       # no quotient of two moments exceeds 1.0014
        # the step refreshed both BF16 copies of the weights: a network given these parameters computes the same bits
        twin = ctl.MLP(widths, seed=1)
        twin.set_params(got)
        assert np.array_equal(net.forward(x), twin.forward(x))
        assert np.array_equal(net.gradient(x, t)[1], twin.gradient(x, t)[1])
        twin.close()
        p = got
    net.close()


# outputs around 1024 and rows around 8192: fused or layer by layer, the same bits for the same row
@pytest.mark.parametrize("widths", [[32, 200, 1024], [32, 200, 1025], [250, 256, 2100]])
def test_inference_does_not_depend_on_the_rows_beside(ctl, gpu, widths):
    print(f"case: mlp rows beside {widths}", flush=True)
    net, p = _init(ctl, widths, seed=3)
    x, _ = _data(widths, 8192, 4)
    whole = net.forward(x)
    for n in (1, 33, 500, 8191):
        assert np.array_equal(net.forward(x[:n]), whole[:n]), n
    want = om.forward(p, widths, x[:200], bf16=True)
    assert np.linalg.norm(whole[:200] - want) <= FWD_REL * np.linalg.norm(want)
    net.close()
