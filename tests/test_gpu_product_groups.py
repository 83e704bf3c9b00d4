"""Products with an element-wise group behind them (csrc/op_epilogue.cpp, kernels/epilogue.h): the group runs on the values that the
product's kernel would store, so every result is bit for bit that of the product and the group one after the other, whose values the
other tests hold against the oracle."""
import ctypes

import numpy as np
import pytest

import jittor_amd as jt
from jittor_amd import _lib as L
from jittor_amd import executor as E

pytestmark = pytest.mark.gpu


def _both(build, fused=1):
    """The graph with its groups behind the products and apart, three times each (captured, replayed, from recorded launches);
    `fused`: how many products take a group along."""
    out = {}
    for on in (True, False):
        jt.flags["enable_product_fusion"] = on
        try:
            before = E.stats["fused_products"]
            for _ in range(3):
                vs = build()
                jt.sync(vs)
                got = [v.raw() for v in vs]
                if on in out:
                    for a, b in zip(out[on], got):
                        assert np.array_equal(a.view(np.uint8), b.view(np.uint8))
                out[on] = [a.copy() for a in got]
            assert (E.stats["fused_products"] - before == 3 * fused) if on else (E.stats["fused_products"] == before)
        finally:
            jt.flags["enable_product_fusion"] = True
    for i, (a, b) in enumerate(zip(out[True], out[False])):
        assert a.shape == b.shape and np.array_equal(a.view(np.uint8), b.view(np.uint8)), "result %d" % i
    return out[True]


def _taken(build):
    """How many groups the graph's kernels take along."""
    before = E.stats["fused_products"]
    jt.sync(build())
    return E.stats["fused_products"] - before


def _var(rng, shape, dt, scale=1.0):
    v = (rng.standard_normal(shape) * scale).astype(np.float32)
    if dt == "bfloat16":
        return jt.from_storage((v.view(np.uint32) >> 16).astype(np.uint16), dt)
    return jt.from_storage(v.astype(L.NP_STORAGE[dt]), dt)


# (images, channels in, out, rows, columns, taps, padding, stride, type): the direct-copy product over pixels (planes of 196, 56 and 64
# values, tiles that end inside one), the convolution kernel at widths of 4, 2 and 1, ragged last rows, groups of 32 channels, first
# layers in float32 and 16 bits, the gathering product whole and in parts, the kernel of one lane a result
CONVS = [(3, 256, 136, 14, 14, 1, 0, 1, "bfloat16"), (5, 128, 256, 8, 7, 1, 0, 1, "float16"), (2, 128, 128, 8, 8, 1, 0, 1, "bfloat16"), (16, 192, 512, 8, 8, 1, 0, 1, "float16"),
         (3, 64, 64, 14, 14, 3, 1, 1, "bfloat16"), (2, 64, 128, 9, 10, 3, 1, 1, "float16"), (2, 32, 64, 17, 20, 3, 1, 1, "bfloat16"), (1, 32, 32, 11, 28, 5, 2, 1, "bfloat16"),
         (2, 3, 24, 64, 64, 7, 3, 2, "float32"), (9, 3, 70, 61, 66, 7, 3, 2, "float32"), (2, 3, 40, 50, 50, 7, 3, 2, "bfloat16"),
         (3, 20, 70, 13, 13, 3, 1, 1, "float32"), (2, 5, 33, 30, 31, 3, 1, 1, "float32"), (4, 60, 100, 11, 13, 3, 1, 1, "bfloat16"), (2, 3, 7, 6, 5, 3, 1, 1, "float32")]


@pytest.mark.parametrize("case", CONVS, ids=str)
def test_convolutions(gpu, case):
    n, c, k, h, w, r, pad, st, dt = case
    rng = np.random.default_rng(7)
    x, wt = _var(rng, [n, c, h, w], dt), _var(rng, [k, c, r, r], dt, (2.0 / (c * r * r)) ** 0.5)
    o = [(d + 2 * pad - r) // st + 1 for d in (h, w)]
    bias, skip, per_image = _var(rng, [k], dt), _var(rng, [n, k] + o, dt), _var(rng, [n, k, 1, 1], dt)
    conv = lambda: jt.nn.conv2d(x, wt, stride=st, padding=pad)
    y, = _both(lambda: [jt.nn.relu(conv())])
    if dt == "float32":
        assert (y == 0).any() and (y > 0).any()
    _both(lambda: [jt.nn.relu(conv() + bias.broadcast([n, k] + o, [0, 2, 3]) + skip)])

    def two():                                                  # two results of other types, a value per image and channel, a scalar
        z = conv() * per_image + 0.25
        return [z > 0.0, z.exp() * 0.5, z.float64()]
    _both(two)


@pytest.mark.parametrize("case", [c for c in CONVS if c[7] == 1], ids=str)
def test_input_gradients(gpu, case):
    n, c, k, h, w, r, pad, st, dt = case
    rng = np.random.default_rng(8)
    x, wt, g = _var(rng, [n, c, h, w], dt), _var(rng, [k, c, r, r], dt, (2.0 / (c * r * r)) ** 0.5), _var(rng, [n, k, h, w], dt)
    mask = _var(rng, [n, c, h, w], dt)

    def step():                                                 # the mask of a relu in front of the convolution, a shortcut around it
        a = jt.nn.relu(x * mask)
        y = jt.nn.conv2d(a, wt, padding=pad)
        return list(jt.grad((y * g).sum() + (a * mask).sum(), [x]))
    _both(step)


@pytest.mark.parametrize("m,k,n", [(128, 128, 128), (256, 512, 260), (1, 64, 8), (130, 72, 66), (257, 1024, 516), (300, 192, 2), (512, 64, 1030)])
@pytest.mark.parametrize("dt", ["float32", "bfloat16", "float16"])
def test_linear(gpu, m, k, n, dt):
    rng = np.random.default_rng(9)
    x, w, b = _var(rng, [m, k], dt), _var(rng, [n, k], dt, k ** -0.5), _var(rng, [n], dt)
    x2, w2, rows = _var(rng, [k, m], dt), _var(rng, [k, n], dt, k ** -0.5), _var(rng, [m, 1], dt)

    # (not where a sum is cut into slices, nor on the kernel without MFMAs)
    for build in (lambda: [jt.nn.relu(jt.nn.linear(x, w, b))], lambda: [jt.nn.matmul(x, w2) * rows],
                  lambda: [jt.nn.linear(x, w, b).sigmoid() * jt.nn.matmul(x, w2)]):
        _both(build, _taken(build))


def test_batches_and_large_tiles(gpu):
    rng = np.random.default_rng(10)
    a, b, s = _var(rng, [6, 128, 64], "bfloat16"), _var(rng, [6, 64, 128], "bfloat16", 0.1), _var(rng, [6, 128, 128], "bfloat16")
    _both(lambda: [jt.nn.bmm(a, b) + s])
    x, w, bias = _var(rng, [3584, 256], "bfloat16"), _var(rng, [3588, 256], "bfloat16", 0.06), _var(rng, [3588], "bfloat16")
    _both(lambda: [jt.nn.relu(jt.nn.linear(x, w, bias))])


@pytest.mark.parametrize("n", [225, 226, 228])
def test_large_tiles_with_rows_that_are_no_vectors(gpu, n, monkeypatch):
    """256 x 256 tiles (asked for by name) whose lanes store one, two or four adjacent results: plain, and with a group."""
    monkeypatch.setenv("MJT_GEMM_DMA", "256")
    rng = np.random.default_rng(14)
    va, vb = _var(rng, [300, 128], "float16"), _var(rng, [n, 128], "float16")
    y, = _both(lambda: [jt.nn.matmul_transpose(va, vb) * 1.0])
    want = va.numpy().astype(np.float64) @ vb.numpy().astype(np.float64).T
    assert np.abs(y.astype(np.float64) - want).max() <= 2.0 ** -11 * np.abs(want).max() * 1.01


def test_values_that_are_not_finite(gpu):
    rng = np.random.default_rng(11)
    x, w = rng.standard_normal((64, 128)).astype(np.float32), rng.standard_normal((128, 128)).astype(np.float32)
    x[3, 5], x[7, 9], x[11, 2] = np.inf, -np.inf, np.nan
    vx, vw = jt.array(x), jt.array(w)
    for dt in ("float32", "bfloat16", "float16"):
        a, b = vx.cast(dt), vw.cast(dt)
        jt.sync([a, b])
        _both(lambda: [jt.nn.relu(jt.nn.matmul(a, b)), ])


# windows that overlap or not, vectors of 4, 2 and 1 elements of a row, a mean's and a maximum's gradient
@pytest.mark.parametrize("shape,k,st,pad,op", [((2, 24, 33, 32), 3, 2, 1, "maximum"), ((3, 16, 18, 22), 2, 2, 0, "maximum"), ((2, 16, 25, 25), 3, 1, 1, "mean"), ((2, 9, 16, 20), 3, 3, 0, "mean")])
@pytest.mark.parametrize("dt", ["float32", "bfloat16", "float16"])
def test_pooling_gradients(gpu, shape, k, st, pad, op, dt):
    """relu, pooling and their gradients: the mask behind the pooling's gradient, read from the relu's result."""
    rng = np.random.default_rng(15)
    x, w = _var(rng, [shape[0], 8] + list(shape[2:]), dt), _var(rng, [shape[1], 8, 3, 3], dt, 0.2)
    o = [(d + 2 * pad - k) // st + 1 for d in shape[2:]]
    g = _var(rng, [shape[0], shape[1]] + o, dt)

    def step():
        y = jt.nn.pool(jt.nn.relu(jt.nn.conv2d(x, w, padding=1)), k, op, pad, st)
        return [y] + list(jt.grad((y * g).sum(), [w]))
    fused = _taken(step)
    assert fused == 2 or (op == "mean" and fused >= 1)
    _both(step, fused)


@pytest.mark.parametrize("dt", ["float32", "bfloat16", "float16"])
def test_masks_of_tiny_and_undefined_values(gpu, dt):
    """y > 0 is x > 0 where x is rounded to y's type already, the smallest numbers and NaN included."""
    tiny = {"float32": [1e-45, -1e-45, 1e-38], "bfloat16": [1e-38, -1e-38, 9.2e-41], "float16": [6e-8, -6e-8, 3e-5]}[dt]
    v = np.array(tiny + [0.0, -0.0, np.inf, -np.inf, np.nan, 1.0, -1.0] + [2.0] * 6, np.float32)
    eye = np.eye(128, dtype=np.float32)
    a = np.zeros((128, 128), np.float32)
    a[:16, 0], a[16:32, 5] = v, v[::-1]
    va, ve, g = jt.array(a).cast(dt), jt.array(eye).cast(dt), jt.array(eye * 3 + 1).cast(dt)
    jt.sync([va, ve, g])

    def step():
        y = jt.nn.relu(jt.nn.matmul(va, ve))
        z = jt.nn.matmul(y, ve)
        return [z] + list(jt.grad((z * g).sum(), [ve, va]))
    _both(step, _taken(step))


@pytest.mark.parametrize("what", ["other", "threshold", "both"])
def test_masks_of_selects_against_other_numbers(gpu, what):
    """One graph with zeros, then with other numbers, captured, replayed and from recorded launches: the mask is that of x > t."""
    rng = np.random.default_rng(16)
    X = rng.integers(-2, 3, (2, 8, 12, 12)).astype(np.float32)
    x, w, g = jt.array(X), _var(rng, [16, 8, 3, 3], "float32"), _var(rng, [2, 16, 12, 12], "float32")
    jt.sync([x, w, g])

    def step(t, b):
        y = jt.ternary(x > jt.array(np.float32([t])), x, jt.array(np.float32([b])))
        gx = jt.grad((jt.nn.conv2d(y, w, padding=1) * g).sum(), x)
        jt.sync([y, gx])
        return y.numpy(), gx.numpy()

    whole = step(-3.0, 0.0)[1]                                   # nothing masked
    assert (whole != 0).all()
    for v in (0.0, 5.0, 0.0, -1.0, 0.0):
        t, b = v if what != "other" else 0.0, v if what != "threshold" else 0.0
        for _ in range(3):
            y, gx = step(t, b)
            assert np.array_equal(y, np.where(X > t, X, np.float32(b))) and np.array_equal(gx, np.where(X > t, whole, 0)), (t, b)


def test_a_product_that_others_read_stays(gpu):
    """A result that is asked for, that a reduce reads too, or that is broadcast, is written as before."""
    rng = np.random.default_rng(12)
    x, w = _var(rng, [64, 128], "float32"), _var(rng, [128, 128], "float32")

    def asked():
        y = jt.nn.matmul(x, w)
        return [y, jt.nn.relu(y)]

    def reduced():
        y = jt.nn.matmul(x, w)
        return [jt.nn.relu(y), y.sum([0])]
    for build in (asked, reduced):
        _both(build, 0)


def test_the_group_leaves_nothing_else_written(gpu):
    """The result lies between guards: stores of whole vectors end where the result ends."""
    lib = L.load()
    rng = np.random.default_rng(13)
    for m, k, n, dt in ((130, 64, 66, "bfloat16"), (257, 128, 132, "float32"), (300, 256, 1028, "bfloat16"), (129, 64, 2, "float16")):
        esz = L.DTYPE_SIZE[dt]
        a, b = _var(rng, [m, k], dt), _var(rng, [k, n], dt)
        guard = 4096
        out = jt.from_storage(np.full([guard * 2 + m * n * esz], 0x5A, np.uint8), "uint8")
        jt.sync([a, b, out], True)
        ta, tb, tc = L.tensor(a.raw_ptr(), dt, [m, k]), L.tensor(b.raw_ptr(), dt, [k, n]), L.tensor(0, dt, [m, n])
        D = L.DTYPE_CODE[dt]
        fv = (L.FusedVar * 2)(L.FusedVar(L.VAR_PRODUCT, D, None), L.FusedVar(L.VAR_OUTPUT, D, out.raw_ptr() + guard))
        fo = (L.FusedOp * 1)(L.FusedOp(L.FOP_UNARY, L.OP_CODE["negative"], (0, 0, 0), 1))
        d = L.FusedDesc(2, (m, n), 2, fv, 1, fo)
        lda, ldb = k * esz % 16, n * esz % 16
        rc = lib.mjt_matmul_then(ctypes.byref(ta), ctypes.byref(tb), ctypes.byref(tc), 0, 0, ctypes.byref(d))
        assert rc in (0, L.ERR_UNSUPPORTED) and (rc == 0 or lda or ldb)
        got = L.d2h(out.raw_ptr(), out.shape, np.uint8)
        assert (got[:guard] == 0x5A).all() and (got[-guard:] == 0x5A).all()
        if rc:
            assert (got == 0x5A).all()
        else:
            plain = jt.from_storage(np.zeros([m, n], L.NP_STORAGE[dt]), dt)
            jt.sync([plain], True)
            tp = L.tensor(plain.raw_ptr(), dt, [m, n])
            L.check(lib.mjt_matmul(ctypes.byref(ta), ctypes.byref(tb), ctypes.byref(tp), 0, 0))
            want = L.d2h(plain.raw_ptr(), plain.shape, L.NP_STORAGE[dt])
            bits = {2: np.uint16, 4: np.uint32}[esz]
            sign = bits(1) << bits(8 * esz - 1)
            assert np.array_equal(got[guard:-guard].view(bits), want.view(bits).reshape(-1) ^ sign)
