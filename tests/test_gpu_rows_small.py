"""Row chains of a few elements run as one kernel, too: a softmax and a cross entropy with their gradients against 64 bits."""
import numpy as np
import pytest

import jittor_amd as jt
from jittor_amd import executor as E

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -24


# a single row, rows of two, fewer elements than lanes, edges of a wave and of a pack
@pytest.mark.parametrize("rows,cols", [(1, 2), (1, 3), (4, 5), (2, 63), (3, 64), (5, 65), (64, 2), (65, 7), (1, 1027), (16, 257)])
def test_softmax(gpu, rows, cols):
    rng = np.random.default_rng(rows * 1000 + cols)
    x, g = (rng.standard_normal((rows, cols)).astype(np.float32) * s for s in (2.0, 1.0))
    vx, vg = jt.array(x), jt.array(g)
    before = E.stats["fused_rows"]
    for _ in range(3):                                         # executed, replayed, from recorded launches
        e = (vx - vx.max([1], keepdims=True)).exp()
        y = e / e.sum([1], keepdims=True)
        dx, = jt.grad((y * vg).sum(), [vx])
        jt.sync([y, dx])
    assert E.stats["fused_rows"] > before
    X, G = x.astype(np.float64), g.astype(np.float64)
    e = np.exp(X - X.max(1, keepdims=True))
    Y = e / e.sum(1, keepdims=True)
    # exp and the subtraction before it: 4 roundings of an exponent of up to |x - max|, the row's sum, the quotient; the gradient's two
    # products cancel, so its error is that of their sizes
    up = (np.abs(X - X.max(1, keepdims=True)).max(1, keepdims=True) + cols + 16) * EPS
    assert (np.abs(y.numpy() - Y) <= up * Y + 1e-38).all()
    assert (np.abs(dx.numpy() - Y * (G - (Y * G).sum(1, keepdims=True))) <= 8 * up * Y * (np.abs(G) + (Y * np.abs(G)).sum(1, keepdims=True)) + 1e-38).all()


@pytest.mark.parametrize("n,classes,width", [(1, 2, 3), (4, 5, 16), (7, 99, 39), (33, 64, 8)])
def test_cross_entropy_step(gpu, n, classes, width):
    """The head of a classifier: linear layer, log softmax, loss and the gradients of weights and bias, against 64 bits."""
    rng = np.random.default_rng(n)
    h, w, b = (rng.standard_normal(s).astype(np.float32) * 0.5 for s in ((n, width), (classes, width), (classes,)))
    onehot = np.eye(classes, dtype=np.float32)[rng.integers(0, classes, n)]
    vh, vw, vb, vo = (jt.array(a) for a in (h, w, b, onehot))
    for _ in range(3):
        logits = jt.nn.linear(vh, vw, vb)
        s = logits - logits.max([1], keepdims=True)
        logp = s - s.exp().sum([1], keepdims=True).log()
        loss = (logp * vo).sum() * (-1.0 / n)
        dw, db = jt.grad(loss, [vw, vb])
        jt.sync([loss, dw, db])
    H, W, B = (a.astype(np.float64) for a in (h, w, b))
    L = H @ W.T + B
    p = np.exp(L - L.max(1, keepdims=True))
    p /= p.sum(1, keepdims=True)
    D = (p - onehot) / n
    up = (np.abs(L).max() * 4 + width + classes + 32) * EPS                     # relative error of a probability
    size = (p + onehot) / n
    assert abs(float(loss.numpy().reshape(-1)[0]) + (np.log(p) * onehot).sum() / n) <= up * (np.abs(np.log(p)) * onehot + 1).sum() / n + up
    assert (np.abs(db.numpy() - D.sum(0)) <= (up + n * EPS) * size.sum(0)).all()
    assert (np.abs(dw.numpy() - D.T @ H) <= (up + n * EPS) * (size.T @ np.abs(H))).all()
