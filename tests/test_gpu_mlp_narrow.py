"""The narrow network's kernels (all layers in one launch) at the edges of their tiling, and the
widths on both sides of the rule that chooses them, against the FP64 oracle with the bounds of
tests/test_gpu_mlp.py: outputs within 2e-5 of max |y|, per-layer gradients within 1e-4 relative in
the 2-norm, the loss within 1e-5 relative.  Mini-batches that wrap around the end of the data give
the gradients of the rows that they hold: a run over wrapped batches equals, bit for bit, a run over
data laid out twice."""
import numpy as np
import pytest

from oracle import mlp_oracle as MO

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def spss():
    import spsslangevinintegration_amd as m
    return m


def _data(n, dims, seed):
    rng = np.random.default_rng(seed)
    x = rng.uniform(-1, 1, (n, dims[0])).astype(np.float32)
    t = np.stack([np.sin(2.0 * x.sum(axis=1) + k) for k in range(dims[-1])], axis=1).astype(np.float32)
    return x, t


@pytest.mark.parametrize("dims,batch,rows", [
    ((6, 128, 128, 128, 2), 257, 32769), ((6, 128, 128, 128, 2), 2, 64), ((1, 1), 1, 1), ((3, 7, 5), 3, 65),
    ((128, 128), 64, 63), ((5, 65, 127, 9), 31, 200), ((6, 16, 17, 15, 33, 8, 3), 300, 129), ((2, 128, 1), 512, 1),
    ((6, 129, 4), 33, 70),               # wider than the narrow kernels
    ((6, 128, 128, 128, 128, 2), 40, 70)])  # weights beyond their LDS
def test_narrow_network_edges(spss, dims, batch, rows):
    print(f"[gpu] mlp dims={dims} batch={batch} rows={rows}", flush=True)
    net = spss.MLP(dims, max_batch=512, seed=9)
    p64 = net.params.astype(np.float64)
    x, t = _data(rows, dims, 1)
    y64 = MO.forward(p64, dims, x.astype(np.float64))[2]
    assert np.max(np.abs(net.predict(x) - y64)) <= 2e-5 * np.max(np.abs(y64))
    x, t = _data(batch, dims, 2)
    loss, g = net.gradients(x, t)
    loss64, g64 = MO.loss_and_grad(p64, dims, x.astype(np.float64), t.astype(np.float64))
    assert abs(loss - loss64) <= 1e-5 * loss64
    for l, (w, b) in enumerate(MO.layout(dims)[0]):
        a, c = g[w:b + dims[l + 1]].astype(np.float64), g64[w:b + dims[l + 1]]
        assert np.linalg.norm(a - c) <= 1e-4 * np.linalg.norm(c), l


def test_narrow_training_wraps_around_the_data(spss):
    dims, n, batch = (6, 40, 33, 2), 101, 64
    print(f"[gpu] mlp training over wrapped batches dims={dims}", flush=True)
    x, t = _data(n, dims, 4)
    out = []
    for reps in (1, batch):  # 64 x 101 rows: the batches never wrap
        net = spss.MLP(dims, max_batch=batch, seed=2)
        net.set_data(np.tile(x, (reps, 1)), np.tile(t, (reps, 1)))
        out.append((net.train(37, batch), net.params))
    np.testing.assert_array_equal(out[0][0], out[1][0])
    np.testing.assert_array_equal(out[0][1], out[1][1])
