"""mjt_fused_rows (csrc/op_rows.cpp, kernels/rows.h) through the front end: chains of element groups and row reduces over one
[rows, columns] space as one kernel, against numpy in float64 and against the same graph run part by part."""
import numpy as np
import pytest

import jittor_amd as jt
import rows_graphs
from jittor_amd import executor as E

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24


def _layernorm(x, gamma, beta, g, n_lead):
    dims = list(range(n_lead, len(x.shape)))
    d = x - x.mean(dims, keepdims=True)
    y = d / ((d * d).mean(dims, keepdims=True) + 1e-5).sqrt() * gamma + beta
    return [y] + list(jt.grad((y * g).sum(), [x, gamma, beta]))


def _softmax(x, g):
    e = (x - x.max([1], keepdims=True)).exp()
    y = e / e.sum([1], keepdims=True)
    return [y] + list(jt.grad((y * g).sum(), [x]))


def _both(build, replays=2):
    """Results fused and part by part, each executed a few times (capture, replay, recorded launches)."""
    out = {}
    for on in (True, False):
        jt.flags["enable_row_fusion"] = on
        try:
            before = E.stats["fused_rows"]
            for _ in range(1 + replays):
                vs = build()
                jt.sync(vs)
                got = [np.asarray(v.numpy(), dtype=np.float64) for v in vs]
                if on in out:
                    for a, b in zip(out[on], got):
                        assert np.array_equal(a, b, equal_nan=True)        # the same sums in the same order every time
                out[on] = got
            assert (E.stats["fused_rows"] > before) == on
        finally:
            jt.flags["enable_row_fusion"] = True
    return out[True], out[False]


# columns: lanes and packs at their edges, odd widths (vectors of one or two), the longest row, a row of one element
@pytest.mark.parametrize("rows,cols", [(33000, 1), (16400, 2), (11000, 3), (1100, 32), (1000, 33), (517, 64), (515, 65), (300, 128), (130, 260), (129, 777), (70, 1000), (67, 1001),
                                       (40, 1028), (17, 2047), (9, 4096), (5, 8200), (3, 16383), (2, 16384)])
def test_layernorm_training_step(gpu, rows, cols):
    rng = np.random.default_rng(rows)
    x, g = rng.standard_normal((rows, cols)).astype(np.float32) * 1.5 + 0.3, rng.standard_normal((rows, cols)).astype(np.float32)
    ga, be = (rng.standard_normal(cols) * 0.2 + 1.0).astype(np.float32), rng.standard_normal(cols).astype(np.float32)
    v = [jt.array(a) for a in (x, ga, be, g)]
    fused, parts = _both(lambda: _layernorm(v[0], v[1], v[2], v[3], 1))
    X, G, GA = (a.astype(np.float64) for a in (x, g, ga))
    d = X - X.mean(1, keepdims=True)
    s = np.sqrt((d * d).mean(1, keepdims=True) + 1e-5)
    h = d / s
    dh = G * GA
    want = [h * GA + be, (dh - dh.mean(1, keepdims=True) - h * (dh * h).mean(1, keepdims=True)) / s, (G * h).sum(0), G.sum(0)]
    # about twenty roundings of terms of the row's size for an element, the sums' magnitudes for theirs; where a row has next to no
    # variance, 1 / s carries them up
    up = 1.0 / s
    bound = [64 * EPS * (np.abs(GA) * up * np.abs(X).max(1, keepdims=True) + np.abs(be)), 256 * EPS * up * (np.abs(dh).max(1, keepdims=True) * (1 + np.abs(h).max(1, keepdims=True) ** 2) * (1 + up)),
             64 * EPS * (np.abs(G) * up * np.abs(X).max(1, keepdims=True)).sum(0), 32 * EPS * np.abs(G).sum(0)]
    for a, b, w, t in zip(fused, parts, want, bound):
        assert a.shape == w.shape and (np.abs(a - w) <= t).all(), float((np.abs(a - w) / t).max())
        assert np.linalg.norm(a - w) <= 1.5 * np.linalg.norm(b - w) + 1e-30 + 4 * EPS * np.linalg.norm(w)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16", "float16"])
@pytest.mark.parametrize("rows,cols", [(1100, 32), (129, 777), (64, 1000), (9, 4096), (2, 16384)])
def test_softmax_with_masks_and_special_values(gpu, dtype, rows, cols):
    """Entries of minus infinity and of the lowest float (masks), rows of nothing else, NaN and infinity: the same elements are finite as
    part by part, and those agree."""
    rng = np.random.default_rng(cols)
    x = (rng.standard_normal((rows, cols)) * 2).astype(np.float32)
    low = -np.float32(3.0e38) if dtype != "float16" else np.float32(-60000)
    x[0, ::3], x[1, :] = -np.inf, low
    if rows > 8:
        x[2, :], x[3, 1], x[4, 2], x[5, ::2] = -np.inf, np.nan, np.inf, low
    g = rng.standard_normal((rows, cols)).astype(np.float32)
    v = [jt.array(a).cast(dtype) for a in (x, g)]
    jt.sync(v)
    fused, parts = _both(lambda: _softmax(*v))
    tol = {"float32": 1e-5, "bfloat16": 2.0 ** -7, "float16": 2.0 ** -9}[dtype]
    for a, b in zip(fused, parts):
        assert np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(np.isinf(a), np.isinf(b))
        ok = np.isfinite(b)
        assert np.abs(a[ok] - b[ok]).max() <= tol * max(1.0, np.abs(b[ok]).max())


@pytest.mark.parametrize("shape,n_lead", [((6, 50, 7, 19), 2), ((6, 50, 7, 19), 1), ((400, 1, 96), 2), ((1, 300, 130), 1), ((3, 4, 5, 700), 3)])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_rows_and_columns_of_several_axes(gpu, shape, n_lead, dtype):
    """Reductions over the last axes, scale and shift over exactly those axes or over the last one only (that group stays outside or is
    broadcast along part of the rows: the parts run), 16-bit results of column sums."""
    rng = np.random.default_rng(sum(shape))
    for tail in {tuple(shape[n_lead:]), tuple(shape[-1:])}:
        x, g = (rng.standard_normal(shape).astype(np.float32) for _ in range(2))
        ga, be = (rng.standard_normal(tail).astype(np.float32) for _ in range(2))
        v = [jt.array(a).cast(dtype) for a in (x, ga, be, g)]
        jt.sync(v)
        out = {}
        for on in (True, False):
            jt.flags["enable_row_fusion"] = on
            try:
                vs = _layernorm(v[0], v[1], v[2], v[3], n_lead)
                jt.sync(vs)
                out[on] = [np.asarray(q.numpy(), dtype=np.float64) for q in vs]
            finally:
                jt.flags["enable_row_fusion"] = True
        for a, b in zip(out[True], out[False]):
            assert np.abs(a - b).max() <= (1e-5 if dtype == "float32" else 2.0 ** -6) * np.abs(b).max()


def test_results_that_others_read_and_later_requests(gpu):
    """A row's statistics asked for beside the result, an intermediate read by an op of another shape, a var left in registers that is
    asked for later; a path that leaves the rows between two reductions (its parts must not run together)."""
    rng = np.random.default_rng(8)
    x = rng.standard_normal((300, 200)).astype(np.float32)
    X = x.astype(np.float64)
    v = jt.array(x)
    m = v.mean([1], keepdims=True)
    d = v - m
    s = (d * d).sum([1], keepdims=True)
    y = d / s.sqrt()
    t = d.transpose([1, 0]).sum([1])                                   # reads d outside the rows
    jt.sync([y, m, t])
    D = X - X.mean(1, keepdims=True)
    S = (D * D).sum(1, keepdims=True)
    assert np.allclose(m.numpy(), X.mean(1, keepdims=True), rtol=1e-5, atol=1e-6) and np.allclose(t.numpy(), D.sum(0), rtol=1e-4, atol=1e-4)
    assert np.allclose(y.numpy(), D / np.sqrt(S), rtol=1e-5, atol=1e-6) and np.allclose(s.numpy(), S, rtol=1e-5)
    # the column sums of one normalisation scale the rows of the next: two kernels in order
    w = jt.array(x)
    e = (w - w.max([1], keepdims=True)).exp()
    p = e / e.sum([1], keepdims=True)
    c = p.sum([0], keepdims=True)
    q = p * c
    r = q / q.sum([1], keepdims=True)
    jt.sync([r])
    P = np.exp(X - X.max(1, keepdims=True))
    P /= P.sum(1, keepdims=True)
    Q = P * P.sum(0, keepdims=True)
    assert np.allclose(r.numpy(), Q / Q.sum(1, keepdims=True), rtol=1e-4, atol=1e-9)


def test_random_graphs_over_rows(gpu):
    """Random DAGs of element ops, row and column reduces with keepdims and their broadcasts, over enough elements for the rows kernel; several
    results at once, against numpy in float64."""
    rng = np.random.default_rng(77)
    before = E.stats["fused_rows"]
    for case in range(40):
        rows, cols = [(520, 64), (130, 257), (40, 1000), (3, 12000), (2000, 17)][case % 5]
        shape = [rows, cols]
        pairs = []
        for _ in range(int(rng.integers(1, 4))):
            a = rng.uniform(-1.5, 1.5, shape).astype(np.float32)
            pairs.append((jt.array(a), a.astype(np.float64)))
        a = rng.uniform(0.5, 1.5, (1, cols)).astype(np.float32)
        pairs.append((jt.array(a), a.astype(np.float64)))

        def pick(full=False):
            cand = [p for p in pairs if not full or list(p[1].shape) == shape]
            return cand[int(rng.integers(len(cand)))]
        for _ in range(int(rng.integers(6, 16))):
            r = rng.random()
            if r < 0.25:
                v, a = pick()
                pairs.append((jt.unary(v, "sigmoid"), 1.0 / (1.0 + np.exp(-a))) if rng.random() < 0.5 else (jt.unary(v, "negative"), -a))
            elif r < 0.6:
                (v, a), (w, b) = pick(), pick()
                op, f = [("add", np.add), ("subtract", np.subtract), ("multiply", np.multiply), ("maximum", np.maximum)][int(rng.integers(4))]
                pairs.append((jt.binary(v, w, op), f(a, b)))
            else:
                v, a = pick(full=True)
                op, f = [("mean", np.mean), ("maximum", np.max), ("minimum", np.min), ("mean", np.mean)][int(rng.integers(4))]
                if rng.random() < 0.2:
                    pairs.append((v.reduce("add", [0], True) * (1.0 / rows), a.mean(0, keepdims=True)))
                else:
                    pairs.append((v.reduce(op, [1], True), f(a, axis=1, keepdims=True)))
        chosen = [pairs[-1 - i] for i in range(min(int(rng.integers(1, 4)), len(pairs)))]
        got = jt.fetch_sync([v for v, _ in chosen])
        for g, (_, want) in zip(got, chosen):
            scale = max(1.0, float(np.abs(want).max()))
            assert list(g.shape) == list(want.shape) and np.allclose(g, want, rtol=2e-4, atol=2e-5 * scale), (case, float(np.abs(g - want).max()), scale)
    assert E.stats["fused_rows"] - before >= 15


@pytest.mark.parametrize("n", [182, 256])
@pytest.mark.parametrize("graph", rows_graphs.GRAPHS + [None])
def test_square_matrices(gpu, graph, n):
    """As many rows as columns, without keepdims: values per row that are read per column.  Terms are of size 0.5 to 1.5, sums of up to n of
    them; a handful of roundings of each, the sums' chains included."""
    rng = np.random.default_rng(n)
    X, e = (rng.uniform(0.5, 1.5, (n, n) if graph else (14, 16, 14, 16)).astype(np.float32), rng.uniform(0.5, 1.5, n).astype(np.float32))
    x, v = jt.array(X), jt.array(e)
    for _ in range(3):                                                 # executed, replayed, as recorded launches
        outs = graph(x, X.astype(np.float64), v, e.astype(np.float64)) if graph else rows_graphs.several_axes(x, X.astype(np.float64))
        for got, (_, want) in zip(jt.fetch_sync([q for q, _ in outs]), outs):
            assert np.abs(got - want).max() <= 64 * EPS * max(n, np.abs(want).max())


def test_more_rows_than_a_launch_takes_at_once(gpu):
    """2^28 + 1024 rows: the workgroups walk on to the rows past the first 2^20 * 256.  Sums of two elements are the same part by part."""
    rng = np.random.default_rng(4)
    a, b = (jt.array(rng.uniform(0.5, 1.5, s).astype(np.float32)).bfloat16() for s in ((1, 1024, 2), (2 ** 18 + 1, 1, 1)))
    x = (a * b).reshape([(2 ** 18 + 1) * 1024, 2])
    jt.sync([x])
    got = {}
    for on in (True, False):
        jt.flags["enable_row_fusion"] = on
        try:
            before = E.stats["fused_rows"]
            got[on] = x - x.max([1], keepdims=True)
            jt.sync([got[on]])
            assert (E.stats["fused_rows"] > before) == on
        finally:
            jt.flags["enable_row_fusion"] = True
    assert float((got[True] - got[False]).abs().max().data[0]) == 0.0 and float(got[True].min().data[0]) < 0.0
