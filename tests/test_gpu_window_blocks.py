"""Pooling on blocks: windows folded from whole 16-byte pieces (kernels/window_fold.h) and their gradients on blocks of rows and columns
(kernels/window_scatter.h with BLOCKS), against the kernels of one output and one row a lane, which are held to the oracle elsewhere: every
result meets its window in the same order, so folds and a maximum's gradient agree bit for bit; the terms of a mean's gradient are products, which one
kernel may round before it adds them and the other not, so it agrees within that rounding."""
import numpy as np
import pytest

import jittor_amd as jt
from jittor_amd import _lib, dtypes

pytestmark = pytest.mark.gpu


def _values(shape, dtype, seed):
    rng = np.random.default_rng(seed)
    if dtype == "int32":
        return jt.array(rng.integers(-1000, 1000, shape).astype(np.int32))
    v = rng.standard_normal(shape)
    v.reshape(-1)[rng.integers(0, v.size, 5)] = [np.inf, -np.inf, 0.0, -0.0, -32768.0]
    if dtype == "bfloat16":
        return jt.from_storage(dtypes.f32_to_bf16_bits(v.astype(np.float32)), dtype)
    return jt.array(v.astype(dtype))



def _same(a, b):
    """The same bits, but for the sign of a NaN, which no operation defines."""
    a, b = (np.where(np.isnan(v), np.nan, v.astype(np.float64)) for v in (a, b))
    return np.array_equal(a, b, equal_nan=True) and np.array_equal(np.signbit(a), np.signbit(b))


def _both(monkeypatch, switch, build):
    """The results with the blocks and without, and the kernel that ran last with them."""
    out = []
    for on in ("1", "0"):
        monkeypatch.setenv(switch, on)
        with jt.flag_scope(enable_replay=0):
            v = build()
            v.sync()
            out.append((v.numpy(), _lib.load().mjt_last_kernel().decode()))
    return out


# kernel, stride, padding, dilation; maps whose results end inside a lane's block, rows shorter than one, single rows and columns
WINDOWS = [(3, 2, 1, 1), (2, 2, 0, 1), (3, 1, 1, 1), (3, 3, 0, 1), (5, 2, 2, 1), (2, 1, 0, 3), (1, 2, 0, 1), (4, 4, 1, 1), (3, 2, 0, 2), (2, 5, 1, 1)]
MAPS = [(1, 1, 8, 8), (2, 3, 7, 16), (3, 1, 13, 24), (1, 2, 33, 40)]


def _cases():
    """Every window on two of the maps, each map with half of the windows (a kernel is built for each)."""
    return [(i, w, MAPS[m]) for i, w in enumerate(WINDOWS) for m in range(len(MAPS)) if (i + m) % 2 == 0]


@pytest.mark.parametrize("dtype,op", [("float32", "maximum"), ("float32", "mean"), ("bfloat16", "maximum"), ("float16", "add"), ("float64", "minimum"), ("int32", "add")])
def test_fold(gpu, monkeypatch, dtype, op):
    took = 0
    for i, (k, s, p, d), shape in _cases():
        o = [(e + 2 * p - d * (k - 1) - 1) // s + 1 for e in shape[2:]]
        if min(o) < 1:
            continue
        x = _values(shape, dtype, i)
        at = ["i0", "i1"] + ["i%d*%d+i%d*%d-%d" % (a, s, a + 2, d, p) for a in (2, 3)]
        (got, name), (want, other) = _both(monkeypatch, "MJT_WINDOW_FOLD",
                                           lambda: x.reindex(list(shape[:2]) + o + [k, k], at, overflow_value=-3.0).reduce(op, [4, 5]))
        assert "window_fold" not in other
        took += "window_fold" in name
        assert _same(got, want), (k, s, p, d, shape)
    assert took >= 8 or dtype in ("bfloat16", "float16")              # (a 16-bit sum is narrowed by a kernel behind the fold)


@pytest.mark.parametrize("dtype,op", [("float32", "maximum"), ("float32", "mean"), ("bfloat16", "maximum"), ("float16", "mean")])
def test_gradient(gpu, monkeypatch, dtype, op):
    took = 0
    for i, (k, s, p, d), shape in _cases():
        o = [(e + 2 * p - (k - 1) - 1) // s + 1 for e in shape[2:]]
        if d != 1 or p >= k or min(o) < 1:
            continue
        x, g = _values(shape, dtype, i), _values(list(shape[:2]) + o, dtype, i + 100)
        (got, name), (want, _) = _both(monkeypatch, "MJT_WINDOW_BLOCKS", lambda: jt.grad((jt.nn.pool(jt.nn.relu(x), k, op, p, s) * g).sum(), x))
        took += "window_scatter" in name
        if op == "maximum":
            assert _same(got, want), (k, s, p, shape)
            continue
        # a mean's terms are products, and whether a product is rounded before it is added is the compiler's choice: of up to
        # ceil(k / s)^2 terms each may differ by half a unit of the sum so far, and a narrowed result by one of its own
        finite = np.isfinite(want)
        assert np.array_equal(finite, np.isfinite(got)) and _same(np.where(finite, 0, got), np.where(finite, 0, want))
        largest = np.abs(g.numpy().astype(np.float64)[np.isfinite(g.numpy())]).max() / (k * k)
        one = {"float32": 0.0, "bfloat16": 2.0 ** -7, "float16": 2.0 ** -10}[dtype]
        a, b = got[finite].astype(np.float64), want[finite].astype(np.float64)
        assert (np.abs(a - b) <= np.ceil(k / s) ** 4 * largest * 2.0 ** -24 + one * np.abs(b) + (2.0 ** -24 if dtype == "float16" else 0)).all(), (k, s, p, shape)
    assert took >= 5
