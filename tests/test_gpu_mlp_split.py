"""Weight gradients of small networks on large batches, whose points are split
over rows of blocks: batches around the size from which they are split and
around a split's unit (2048 points), and networks of few and of more blocks."""
import numpy as np
import pytest

from oracle import mlp_oracle as MO
from tmp_amd import mlp

pytestmark = pytest.mark.gpu

SHAPES = [(3, 64, 2, 1), (128, 64, 2, 16), (3, 192, 2, 4), (73, 256, 3, 4), (20, 64, 8, 2)]
POINTS = [16256, 16384, 16385, 18560, 40000]


def _net(nin, width, nlayer, nout):
    w, b = MO.init_params(nin, width, nlayer, nout, 5)
    b = (b + np.random.default_rng(6).normal(0, 0.05, b.size)).astype(np.float32)
    g = mlp.MLP(nin, width, nlayer, nout)
    g.set_params(w, b)
    return g, w, b


@pytest.mark.parametrize("n", POINTS)
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_every_point_counts_once(shape, n):
    """Targets are the network's own outputs but for 64 points, first of all,
    then in the middle, then the last: the gradients are those of these points
    alone, scaled (bars of test_gpu_mlp_shapes: the output gradients are rounded
    to BF16 at another scale)."""
    g, _, _ = _net(*shape)
    rng = np.random.default_rng(7)
    x = rng.normal(size=(n, shape[0])).astype(np.float32)
    own = g.predict(x)
    for a in (0, n // 2, n - 64):
        y = own.copy()
        y[a:a + 64] += rng.normal(size=(64, shape[3])).astype(np.float32)
        loss, dw, db = g.gradients(x, y)
        ref, rw, rb = g.gradients(x[a:a + 64], y[a:a + 64])
        k = 64 / n
        assert abs(loss - ref * k) <= 1e-3 * ref * k
        assert np.linalg.norm(dw - rw * k) <= 2e-2 * np.linalg.norm(rw * k)
        assert np.linalg.norm(db - rb * k) <= 2e-2 * np.linalg.norm(rb * k)


@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_sum_over_splits(shape):
    """32768 points against four quarters, which are not split: the mean's
    factor is a power of two, so only the order of the FP32 sums differs (chunks
    of 256 points: under 128 additions of 2^-24 each, of sums with random signs)."""
    g, _, _ = _net(*shape)
    rng = np.random.default_rng(8)
    x = rng.normal(size=(32768, shape[0])).astype(np.float32)
    y = rng.normal(size=(32768, shape[3])).astype(np.float32)
    got = g.gradients(x, y)
    parts = [g.gradients(x[a:a + 8192], y[a:a + 8192]) for a in range(0, 32768, 8192)]
    for i, bar in ((1, 128 * 2.0 ** -24), (2, 128 * 2.0 ** -24)):
        ref = np.mean([p[i].astype(np.float64) for p in parts], axis=0)
        size = np.sqrt(np.mean([np.sum(p[i].astype(np.float64) ** 2) for p in parts]))
        assert np.linalg.norm(got[i] - ref) <= bar * size
    again = g.gradients(x, y)
    assert all(np.array_equal(a, b) for a, b in zip(got, again))


@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_adam_on_split_gradients(shape):
    """One step from no moments is lr g / (|g| + eps), on the gradients that
    gradients() returns for the same batch.  The kernel's FP32 moments and their
    corrections (1 - 0.999^t has 1.3e-5 of its value in rounding, half of that
    after the root) leave 2e-5 of lr, the update one rounding of the parameter."""
    n, lr = 16400, 1e-3
    g, w, b = _net(*shape)
    rng = np.random.default_rng(9)
    x = rng.normal(size=(n, shape[0])).astype(np.float32)
    y = rng.normal(size=(n, shape[3])).astype(np.float32)
    loss, dw, db = g.gradients(x, y)
    g.set_data(x, y)
    got = g.train_epoch(np.arange(n), n, lr)
    d, p = np.concatenate([dw, db]).astype(np.float64), np.concatenate([w, b]).astype(np.float64)
    want = p - lr * d / (np.abs(d) + 1e-8)
    err = np.abs(np.concatenate(g.get_params()) - want)
    assert np.all(err <= 2e-5 * lr + 2.0 ** -23 * np.abs(want))
    assert abs(got - loss) <= 1e-6 * loss
