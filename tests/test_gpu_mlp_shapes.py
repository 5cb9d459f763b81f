"""The network kernels over the shapes they take: widths of each instance,
two layers, more layers than LDS holds rows of, input counts on both sides of
the first layer's padding, and point counts around a block (32), a step of the
weight gradient (128) and a chunk (256).  Bars as in test_gpu_mlp: the oracle
rounds the same operands to BF16 but accumulates in float64."""
import numpy as np
import pytest

from oracle import mlp_oracle as MO
from tmp_amd import mlp

pytestmark = pytest.mark.gpu

SHAPES = [  # nin, width, nlayer, nout, points
    (1, 64, 2, 1, 1),
    (64, 64, 3, 16, 31),
    (65, 128, 2, 4, 33),
    (128, 192, 4, 3, 129),
    (73, 256, 8, 4, 257),
    (72, 256, 12, 4, 385),
    (20, 64, 40, 2, 127),
]


def _net(nin, width, nlayer, nout):
    w, b = MO.init_params(nin, width, nlayer, nout, 5)
    b = (b + np.random.default_rng(6).normal(0, 0.05, b.size)).astype(np.float32)
    g = mlp.MLP(nin, width, nlayer, nout)
    g.set_params(w, b)
    return g, w, b


@pytest.mark.parametrize("nin,width,nlayer,nout,n", SHAPES)
def test_shapes_match_oracle(nin, width, nlayer, nout, n):
    g, w, b = _net(nin, width, nlayer, nout)
    rng = np.random.default_rng(7)
    x = rng.normal(size=(n, nin)).astype(np.float32)
    y = rng.normal(size=(n, nout)).astype(np.float32)
    o = MO.MLP(nin, width, nlayer, nout, w, b, bf16=True)
    ref, _ = o.forward(x.astype(np.float64))
    assert np.max(np.abs(g.predict(x) - ref)) <= 1e-2 * np.max(np.abs(ref))
    loss, dw, db = g.gradients(x, y)
    lo, gW, gb = o.loss_grads(x.astype(np.float64), y.astype(np.float64))
    rw, rb = o.flat(gW, gb)
    assert abs(loss - lo) <= 1e-3 * lo
    assert np.linalg.norm(dw - rw) <= 2e-2 * np.linalg.norm(rw)
    assert np.linalg.norm(db - rb) <= 2e-2 * np.linalg.norm(rb)


@pytest.mark.parametrize("n,batch", [(300, 512), (257, 256), (256, 128)])
def test_epoch_is_adam_on_the_gradients(n, batch):
    """An epoch equals gradients() of each batch followed by Adam in numpy:
    parameters to rounding of the update (1e-5 of the step size)."""
    nin, width, nlayer, nout, lr = 20, 64, 3, 2, 1e-3
    g, w, b = _net(nin, width, nlayer, nout)
    rng = np.random.default_rng(8)
    x = rng.normal(size=(n, nin)).astype(np.float32)
    y = rng.normal(size=(n, nout)).astype(np.float32)
    perm = rng.permutation(n)
    g.set_data(x, y)
    loss = g.train_epoch(perm, batch, lr)
    h, _, _ = _net(nin, width, nlayer, nout)
    p = np.concatenate([w, b]).astype(np.float64)
    m1, m2, losses = np.zeros_like(p), np.zeros_like(p), []
    for t, a in enumerate(range(0, n, batch), 1):
        j = perm[a:a + batch]
        h.set_params(p[:w.size].astype(np.float32), p[w.size:].astype(np.float32))
        lb, dw, db = h.gradients(x[j], y[j])
        losses.append(lb)
        d = np.concatenate([dw, db]).astype(np.float64)
        m1 = 0.9 * m1 + 0.1 * d
        m2 = 0.999 * m2 + 0.001 * d * d
        p -= lr * (m1 / (1 - 0.9 ** t)) / (np.sqrt(m2 / (1 - 0.999 ** t)) + 1e-8)
    gw, gb = g.get_params()
    # FP32 moments and updates: a few 1e-7 of the step, and of the parameter itself
    err = np.abs(np.concatenate([gw, gb]) - p)
    assert np.max(err) <= 1e-2 * lr + 2e-7
    assert np.linalg.norm(err) <= 1e-3 * lr * np.sqrt(p.size)
    assert abs(loss - np.mean(losses)) <= 1e-5 * abs(loss)
