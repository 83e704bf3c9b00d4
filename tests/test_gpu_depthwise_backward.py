"""Both gradients of a depthwise convolution from one kernel (csrc/kernels/conv_depthwise.h, MODE 2)."""
import ctypes

import numpy as np
import pytest

import jittor_amd as jt
from jittor_amd import _lib as L

pytestmark = pytest.mark.gpu

# strips past the last row and column, rows of a plane as tiles, several small planes a workgroup, one slice and many, 1 to 49 taps, padding
# from none to the taps' reach, vectors of 4, 2 and 1
CASES = [((32, 6, 20, 24), (3, 3), (1, 1)), ((5, 3, 7, 7), (3, 3), (1, 1)), ((3, 4, 9, 10), (5, 5), (2, 2)), ((2, 3, 130, 100), (3, 3), (1, 0)), ((40, 2, 13, 11), (7, 7), (3, 6)),
         ((520, 3, 5, 6), (3, 3), (1, 1)), ((4, 130, 14, 14), (3, 2), (0, 1)), ((1, 2, 1, 1), (3, 3), (1, 1)), ((9, 3, 33, 4), (1, 5), (0, 4)), ((70, 8, 16, 16), (3, 3), (2, 2))]


def _store(a, dt):
    a = a.astype(np.float32)
    return jt.from_storage((a.view(np.uint32) >> 16).astype(np.uint16) if dt == "bfloat16" else a.astype(L.NP_STORAGE[dt]), dt)


def _run(xs, rs, pad, dt, odt, fill):
    """(dx, dw) from the one kernel and from the two."""
    n, c, h, w = xs
    (r, s), (ph, pw) = rs, pad
    ys = [n, c, h + 2 * ph - r + 1, w + 2 * pw - s + 1]
    x, dy, wt = (_store(a, dt) for a in fill((xs, ys, [c, 1, r, s])))
    outs = [jt.from_storage(np.full(q, 7, L.NP_STORAGE[odt]), odt) for q in (xs, [c, 1, r, s], xs, [c, 1, r, s])]
    jt.sync([x, dy, wt] + outs, True)
    tx, td, tw, a, b, a2, b2 = (ctypes.byref(L.tensor(v.raw_ptr(), v.dtype, v.shape)) for v in [x, dy, wt] + outs)
    p = L.ConvParams(1, 1, ph, pw, 1, 1)
    lib = L.load()
    L.check(lib.mjt_conv2d_meta_backward_depthwise(tx, td, tw, a, b, ctypes.byref(p), c))
    assert "_backward_direct_" in L.last_kernel()
    rc = lib.mjt_conv2d_meta_dgrad_depthwise(td, tw, a2, ctypes.byref(p), c)
    assert rc == 0
    L.check(lib.mjt_conv2d_meta_wgrad_grouped(tx, td, b2, ctypes.byref(p), c))
    return [L.d2h(v.raw_ptr(), v.shape, L.NP_STORAGE[odt]) for v in outs]


@pytest.mark.parametrize("dt,odt", [("float32", "float32"), ("bfloat16", "bfloat16"), ("float16", "float32")])
@pytest.mark.parametrize("xs,rs,pad", CASES, ids=str)
def test_equals_the_two_kernels(gpu, xs, rs, pad, dt, odt):
    """Whole numbers whose products and sums are exact in float32 (and their results rounded alike): the same bits."""
    rng = np.random.default_rng(3)
    dx, dw, dx2, dw2 = _run(list(xs), rs, pad, dt, odt, lambda shapes: [rng.integers(-3, 4, q) for q in shapes])
    assert np.array_equal(dx, dx2) and np.array_equal(dw, dw2)
    assert np.any(dw2 != 0) or xs[2] * xs[3] == 1


@pytest.mark.parametrize("what", ["x", "dy"])
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("xs,pad", [((3, 4, 7, 7), (1, 1)), ((4, 4, 20, 24), (1, 1)), ((2, 4, 130, 100), (1, 2)), ((3, 4, 6, 9), (0, 0))])
def test_values_that_are_not_finite(gpu, xs, pad, what, value):
    """At corners, borders and inside: in the sums that contain them, as in the two kernels, and in no other."""
    rng = np.random.default_rng(4)
    h, w = xs[2:]
    oh, ow = h + 2 * pad[0] - 2, w + 2 * pad[1] - 2
    rows, cols = (h, w) if what == "x" else (oh, ow)
    for at in ((0, 0), (rows - 1, cols - 1), (0, cols // 2), (rows // 2, cols - 1), (rows // 2, cols // 2)):
        def fill(shapes):
            v = [rng.integers(1, 5, q).astype(np.float32) for q in shapes]
            v[0 if what == "x" else 1][1, 2][at] = value
            return v
        dx, dw, dx2, dw2 = _run(list(xs), (3, 3), pad, "float32", "float32", fill)
        assert np.array_equal(dx, dx2, equal_nan=True) and np.array_equal(dw, dw2, equal_nan=True), at


def test_what_it_does_not_take(gpu):
    x = jt.zeros([2, 4, 8, 8])
    jt.sync([x], True)
    t = lambda shape: ctypes.byref(L.tensor(x.raw_ptr(), "float32", shape))
    call = lambda ys, ws, p, g: L.load().mjt_conv2d_meta_backward_depthwise(t([2, 4, 8, 8]), t(ys), t(ws), t([2, 4, 8, 8]), t(ws), ctypes.byref(L.ConvParams(*p)), g)
    assert call([2, 4, 4, 4], [4, 1, 3, 3], (2, 2, 1, 1, 1, 1), 4) == L.ERR_UNSUPPORTED
    assert call([2, 4, 6, 6], [4, 1, 3, 3], (1, 1, 1, 1, 2, 2), 4) == L.ERR_UNSUPPORTED
    assert call([2, 4, 8, 8], [4, 2, 3, 3], (1, 1, 1, 1, 1, 1), 2) == L.ERR_UNSUPPORTED
    assert call([2, 4, 14, 14], [4, 1, 3, 3], (1, 1, 4, 4, 1, 1), 4) == L.ERR_UNSUPPORTED
    assert call([2, 4, 7, 8], [4, 1, 3, 3], (1, 1, 1, 1, 1, 1), 4) == L.ERR_INVALID


def test_the_graph_of_a_training_step(gpu):
    rng = np.random.default_rng(5)
    x, w, g = (jt.array(rng.standard_normal(q).astype(np.float32)) for q in ([8, 16, 20, 20], [16, 1, 3, 3], [8, 16, 20, 20]))

    def step(scale):
        a = x * scale
        y = jt.nn.conv2d(a, w, padding=1, groups=16)
        return list(jt.grad((y * g).sum(), [x, w]))
    for scale in (1.0, 2.0, 0.5):
        got = step(scale)
        jt.sync(got)
        xp = np.pad(x.numpy().astype(np.float64) * scale, ((0, 0), (0, 0), (1, 1), (1, 1)))
        dw, dxp = np.zeros([16, 1, 3, 3]), np.zeros(xp.shape)
        gv, wv = g.numpy().astype(np.float64), w.numpy().astype(np.float64)
        for r in range(3):
            for s in range(3):
                dw[:, 0, r, s] = (gv * xp[:, :, r:r + 20, s:s + 20]).sum((0, 2, 3))
                dxp[:, :, r:r + 20, s:s + 20] += gv * wv[:, 0, r, s][None, :, None, None] * scale
        assert np.abs(got[1].numpy() - dw).max() <= 3200 * 2.0 ** -24 * np.abs(xp).max() * np.abs(gv).max()
        assert np.abs(got[0].numpy() - dxp[:, :, 1:-1, 1:-1]).max() <= 16 * 2.0 ** -24 * np.abs(dxp).max()
