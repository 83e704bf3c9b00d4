"""The weight gradient from windows that lie in LDS (csrc/kernels/conv_wgrad_window.h): pieces of 8 pixels, column phases, stages of rows
and of images, remainders of channels, and infinities at the places that are cleared."""
import ctypes

import numpy as np
import pytest

import jittor_amd as jt
from jittor_amd import _lib as L

pytestmark = pytest.mark.gpu


def _operand(v, dt):
    if dt == "float16":
        h = v.astype(np.float16)
        return jt.from_storage(h, dt), h.astype(np.float64)
    bits = (v.astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)
    return jt.from_storage(bits, dt), (bits.astype(np.uint32) << 16).view(np.float32).astype(np.float64)


def _call(x, dy, rs, p, odt):
    out = jt.from_storage(np.full((dy.shape[1], x.shape[1], *rs), 7, L.NP_STORAGE[odt]), odt)
    jt.sync([out], True)
    tx, td, tw = (L.tensor(v.raw_ptr(), v.dtype, v.shape) for v in (x, dy, out))
    cp = L.ConvParams(*p)
    L.check(L.load().mjt_conv2d_meta_wgrad(ctypes.byref(tx), ctypes.byref(td), ctypes.byref(tw), ctypes.byref(cp)))
    assert "_window_" in L.last_kernel(), L.last_kernel()
    got = L.d2h(out.raw_ptr(), out.shape, L.NP_STORAGE[odt])
    return (got.astype(np.uint32) << 16).view(np.float32).astype(np.float64) if odt == "bfloat16" else got.astype(np.float64)


def _want(xf, df, rs, p):
    sh, sw, ph, pw, dh, dw = p
    oh, ow = df.shape[2:]
    xp = np.pad(xf, ((0, 0), (0, 0), (ph, ph), (pw, pw)))
    want = np.zeros((df.shape[1], xf.shape[1], *rs))
    a = np.ascontiguousarray(df.transpose(1, 0, 2, 3)).reshape(df.shape[1], -1)
    for r in range(rs[0]):
        for s in range(rs[1]):
            patch = xp[:, :, r * dh:r * dh + (oh - 1) * sh + 1:sh, s * dw:s * dw + (ow - 1) * sw + 1:sw]
            want[:, :, r, s] = a @ np.ascontiguousarray(patch.transpose(0, 2, 3, 1)).reshape(-1, xf.shape[1])
    return want


CASES = [
    dict(x=(9, 500, 7, 7), k=520, rs=(3, 3), p=(1, 1, 1, 1, 1, 1)),       # rows of one piece, pairs of images and one left over, ragged channels
    dict(x=(16, 512, 14, 14), k=512, rs=(3, 3), p=(1, 1, 1, 1, 1, 1)),    # whole images, rows of two pieces, the second short by two
    dict(x=(3, 128, 14, 14), k=64, rs=(3, 3), p=(1, 1, 1, 1, 1, 1)),      # half images
    dict(x=(2, 128, 13, 28), k=64, rs=(3, 3), p=(1, 1, 1, 1, 1, 1)),      # four pieces; stages of three rows, the last of one
    dict(x=(2, 128, 16, 64), k=64, rs=(3, 3), p=(1, 1, 1, 1, 1, 1)),      # eight whole pieces
    dict(x=(20, 310, 27, 26), k=290, rs=(3, 3), p=(2, 2, 1, 1, 1, 1)),    # stride 2: two column phases, an odd map, results by single floats
    dict(x=(64, 256, 28, 28), k=256, rs=(3, 3), p=(2, 2, 1, 1, 1, 1)),
    dict(x=(30, 400, 9, 9), k=390, rs=(3, 3), p=(1, 2, 1, 2, 1, 2)),      # dilation on stride 2: one phase is not read
    dict(x=(2, 128, 10, 16), k=128, rs=(3, 3), p=(1, 1, 2, 2, 2, 2)),
    dict(x=(2, 128, 12, 12), k=128, rs=(1, 2), p=(1, 1, 0, 0, 1, 2)),     # two taps, no padding
    dict(x=(3, 128, 9, 8), k=64, rs=(9, 1), p=(1, 1, 4, 0, 1, 1)),        # nine rows of one tap
    dict(x=(2, 128, 11, 30), k=64, rs=(3, 3), p=(1, 1, 0, 2, 1, 1)),      # more padding than taps need
    dict(x=(30, 400, 9, 5), k=390, rs=(3, 3), p=(1, 1, 1, 1, 1, 1)),      # rows shorter than a piece
    dict(x=(5, 128, 5, 6), k=128, rs=(3, 3), p=(3, 1, 1, 1, 1, 1)),       # vertical stride 3
    dict(x=(1, 128, 1, 8), k=64, rs=(1, 3), p=(1, 1, 0, 1, 1, 1)),        # a single row
]


@pytest.mark.parametrize("case", CASES)
def test_window_weight_gradient(gpu, case):
    """Products are exact and sums float32: 1e-4 of the sums of magnitudes (16 products a rounding: at most 784 + 16 slices of them, 2^-24
    each, 5e-5), and one rounding (or truncation) for a result of 16 bits."""
    rng = np.random.default_rng(17)
    n, c, h, w = case["x"]
    (r, s), (sh, sw, ph, pw, dh, dw) = case["rs"], case["p"]
    oh, ow = (h + 2 * ph - dh * (r - 1) - 1) // sh + 1, (w + 2 * pw - dw * (s - 1) - 1) // sw + 1
    for dt in ("bfloat16", "float16"):
        x, xf = _operand(rng.standard_normal((n, c, h, w)), dt)
        dy, df = _operand(rng.standard_normal((n, case["k"], oh, ow)), dt)
        jt.sync([x, dy], True)
        want, mag = _want(xf, df, case["rs"], case["p"]), _want(np.abs(xf), np.abs(df), case["rs"], case["p"])
        for odt in ("float32", dt):
            got = _call(x, dy, case["rs"], case["p"], odt)
            bound = 1e-4 * mag + (0 if odt == "float32" else np.abs(want) * (2.0 ** -7 if dt == "bfloat16" else 2.0 ** -10))
            assert (np.abs(got - want) <= bound).all(), float(np.abs(got - want).max())


@pytest.mark.parametrize("case", [CASES[i] for i in (0, 2, 3, 5, 7, 12)])
def test_window_weight_gradient_keeps_infinities_in_their_taps(gpu, case):
    """An infinity at a border of x reaches exactly the taps that see it, although what lies behind a row's last pixel shares its piece."""
    rng = np.random.default_rng(18)
    n, c, h, w = case["x"]
    (r, s), (sh, sw, ph, pw, dh, dw) = case["rs"], case["p"]
    oh, ow = (h + 2 * ph - dh * (r - 1) - 1) // sh + 1, (w + 2 * pw - dw * (s - 1) - 1) // sw + 1
    v = rng.integers(1, 9, (n, c, h, w)).astype(np.float32)
    g = rng.integers(1, 9, (n, case["k"], oh, ow)).astype(np.float32)          # exact, no sum cancels
    places = [(0, 0), (0, w - 1), (h - 1, 0), (h - 1, w - 1), (h // 2, w - 1), (h - 1, w // 2)]
    for i, (y, z) in enumerate(places):
        v[i % n, 3 * i + 1, y, z] = np.inf
    x, xf = _operand(v, "bfloat16")
    dy, df = _operand(g, "bfloat16")
    jt.sync([x, dy], True)
    got = _call(x, dy, case["rs"], case["p"], "float32")
    with np.errstate(invalid="ignore"):
        xp = np.pad(xf, ((0, 0), (0, 0), (ph, ph), (pw, pw)))
    seen = np.zeros((c, r, s), bool)
    for a in range(r):
        for b in range(s):
            patch = xp[:, :, a * dh:a * dh + (oh - 1) * sh + 1:sh, b * dw:b * dw + (ow - 1) * sw + 1:sw]
            seen[:, a, b] = np.isinf(patch).any((0, 2, 3))
    assert seen.any() and not seen.all()
    assert np.array_equal(np.isinf(got), np.broadcast_to(seen, got.shape)) and not np.isnan(got).any()
    want = _want(np.where(np.isinf(xf), 0, xf), df, case["rs"], case["p"])
    keep = ~np.broadcast_to(seen, got.shape)
    assert np.array_equal(got[keep], want[keep])                               # whole numbers below 2^24
