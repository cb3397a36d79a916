"""Training of the closure network: the gradient against the oracle
(oracle/mlp.py) at row counts around the row tiles (16) and the gradient's
chunks (64 rows, then a 32nd of the batch), and mini-batches named by row
indices against the same rows laid out in order."""
import numpy as np
import pytest

import mlp as MO
from dg_amd import closure, hip

pytestmark = pytest.mark.gpu


def network(seed):
    rng = np.random.default_rng(seed)
    m = closure.MLP(0)
    p = np.concatenate([rng.normal(0, 0.2, int(np.prod(s))) for _, s in MO.SHAPES]).astype(np.float32)
    xm = rng.normal(0, 0.1, MO.NF).astype(np.float32)
    xs = rng.uniform(0.5, 2.0, MO.NF).astype(np.float32)
    ys = rng.uniform(0.5, 2.0, MO.NO).astype(np.float32)
    m.set_params(p)
    m.set_scaling(xm, xs, ys)
    return m, p, xm.astype(np.float64), xs.astype(np.float64), ys.astype(np.float64)


def rows_of(n, seed):
    rng = np.random.default_rng(seed)
    return (rng.normal(0, 1, (n, MO.NF)).astype(np.float32), rng.normal(0, 1, (n, MO.NO)).astype(np.float32))


@pytest.mark.parametrize("rows", [2081, 2049, 2048, 130, 65, 64, 17, 16, 15, 1])
def test_gradient_against_the_oracle(rows):
    print(f"closure gradient, {rows} rows", flush=True)
    m, p, xm, xs, ys = network(rows)
    X, Y = rows_of(rows, rows + 1)
    g, loss = m.gradient(hip.Buffer.from_array(X, np.float32), hip.Buffer.from_array(Y, np.float32), rows)
    m.close()
    lref, gref = MO.loss_and_grad(p, X, Y, xm, xs, ys)
    # FP32 activations and sums of up to some thousand terms: the bars of the
    # whole network's gradient (1e-5 and 1e-4 of a block's largest entry)
    assert abs(loss - lref) < 1e-5 * lref
    o = 0
    for name, shp in MO.SHAPES:
        n = int(np.prod(shp))
        a, b = g[o:o + n], gref[o:o + n]
        assert np.max(np.abs(a - b)) < 1e-4 * np.max(np.abs(b)), name
        o += n


@pytest.mark.parametrize("batch,batches", [(17, 3), (64, 2), (500, 2)])
@pytest.mark.parametrize("noise", [0.0, 0.05])
def test_indexed_batches_match_the_rows_in_order(batch, batches, noise):
    print(f"closure training, {batches} x {batch}, noise {noise}", flush=True)
    n = batch * batches
    X, Y = rows_of(n, 7)
    idx = np.random.default_rng(5).integers(-2, n + 2, n).astype(np.int32)       # also out of range: clamped
    order = np.clip(idx, 0, n - 1)
    out = []
    for x, y, i in ((X, Y, idx), (X[order], Y[order], np.arange(n, dtype=np.int32))):
        m = network(11)[0]
        loss = m.train(hip.Buffer.from_array(x, np.float32), hip.Buffer.from_array(y, np.float32), n,
                       hip.Buffer.from_array(i, np.int32), batch, 1e-3, noise)
        out.append((loss, m.params()))
        m.close()
    assert np.isfinite(out[0][0]) and out[0][0] == out[1][0]
    assert np.array_equal(out[0][1], out[1][1])
    assert np.any(out[0][1] != network(11)[1])
