"""The weight gradient of float32 convolutions of images with few channels from windows in LDS (csrc/kernels/conv_stem_wgrad.h): loads of 4, 2
and 1 values of either operand, remainders of channels, columns, rows and pixels, and operands at the ends of the range."""
import ctypes

import numpy as np
import pytest

import jittor_amd as jt
from jittor_amd import _lib as L

pytestmark = pytest.mark.gpu


def _call(x, dy, k, rs, p):
    vx, vd = jt.from_storage(x.astype(np.float32), "float32"), jt.from_storage(dy.astype(np.float32), "float32")
    out = jt.from_storage(np.full([k, x.shape[1], *rs], 7, np.float32), "float32")
    jt.sync([vx, vd, out], True)
    tx, td, tw = (L.tensor(v.raw_ptr(), "float32", v.shape) for v in (vx, vd, out))
    cp = L.ConvParams(*p)
    L.check(L.load().mjt_conv2d_meta_wgrad(ctypes.byref(tx), ctypes.byref(td), ctypes.byref(tw), ctypes.byref(cp)))
    assert "_stem_" in L.last_kernel(), L.last_kernel()
    return L.d2h(out.raw_ptr(), out.shape, np.float32).astype(np.float64)


def _extents(case):
    (n, c, h, w), (r, s), (sh, sw, ph, pw, dh, dw) = case["x"], case["rs"], case["p"]
    return (n, case["k"], (h + 2 * ph - dh * (r - 1) - 1) // sh + 1, (w + 2 * pw - dw * (s - 1) - 1) // sw + 1)


def _want(x, dy, rs, p):
    sh, sw, ph, pw, dh, dw = p
    oh, ow = dy.shape[2:]
    xp = np.pad(x.astype(np.float64), ((0, 0), (0, 0), (ph, ph), (pw, pw)))
    a = np.ascontiguousarray(dy.astype(np.float64).transpose(1, 0, 2, 3)).reshape(dy.shape[1], -1)
    want = np.zeros((dy.shape[1], x.shape[1], *rs))
    for r in range(rs[0]):
        for s in range(rs[1]):
            patch = xp[:, :, r * dh:r * dh + (oh - 1) * sh + 1:sh, s * dw:s * dw + (ow - 1) * sw + 1:sw]
            want[:, :, r, s] = a @ np.ascontiguousarray(patch.transpose(0, 2, 3, 1)).reshape(-1, x.shape[1])
    return want


CASES = [
    dict(x=(4, 3, 224, 224), k=64, rs=(7, 7), p=(2, 2, 3, 3, 1, 1)),
    dict(x=(48, 3, 65, 65), k=50, rs=(7, 7), p=(2, 2, 3, 3, 1, 1)),       # odd rows: single values; the last channels and pixels are short
    dict(x=(16, 3, 63, 92), k=20, rs=(7, 7), p=(2, 2, 2, 2, 1, 1)),       # one half of the channels, four groups of steps; pairs of dy
    dict(x=(16, 3, 50, 66), k=70, rs=(7, 7), p=(1, 2, 0, 0, 1, 1)),       # no padding, vertical stride 1, two blocks of channels, pairs of x
    dict(x=(64, 3, 64, 96), k=33, rs=(4, 8), p=(3, 2, 1, 2, 2, 1)),       # dilated rows, vertical stride 3; columns end inside a tile
]


@pytest.mark.parametrize("case", CASES)
def test_stem_weight_gradient(gpu, case):
    """Six roundings for 16 pixels and one for each slice, 2^-24 of the sum of magnitudes each; in practice they hardly add up."""
    rng = np.random.default_rng(41)
    ys = _extents(case)
    x, dy = rng.standard_normal(case["x"]).astype(np.float32), rng.standard_normal(ys).astype(np.float32)
    got, want, mag = _call(x, dy, case["k"], case["rs"], case["p"]), _want(x, dy, case["rs"], case["p"]), _want(np.abs(x), np.abs(dy), case["rs"], case["p"])
    assert (np.abs(got - want) <= (ys[0] * ys[2] * ys[3] * 6 / 16 + 512) * 2.0 ** -24 * mag).all()
    assert np.linalg.norm(got - want) <= 2e-6 * np.linalg.norm(want), float(np.linalg.norm(got - want) / np.linalg.norm(want))


@pytest.mark.parametrize("case", CASES[1:3])
def test_stem_weight_gradient_keeps_infinities_in_their_taps(gpu, case):
    """Positive whole numbers and infinities at the corners of x: taps that see one are infinite, all others exact, nothing is NaN."""
    rng = np.random.default_rng(42)
    n, c, h, w = case["x"]
    ys = _extents(case)
    x, dy = rng.integers(1, 5, case["x"]).astype(np.float32), rng.integers(1, 5, ys).astype(np.float32)
    x[0, 0, 0, 0] = x[1, c - 1, h - 1, w - 1] = np.inf
    got = _call(x, dy, case["k"], case["rs"], case["p"])
    seen = _want(np.isinf(x).astype(float), np.ones_like(dy), case["rs"], case["p"]) > 0
    assert seen.any() and not seen.all()
    assert np.array_equal(np.isinf(got), seen) and not np.isnan(got).any()
    want = _want(np.where(np.isinf(x), 0, x), dy, case["rs"], case["p"])
    assert want.max() < 2 ** 24 and np.array_equal(got[~seen], want[~seen])


@pytest.mark.parametrize("xscale,dscale", [(1e-33, 1e-2), (1e-20, 1e-19), (1e16, 1e17), (1e-2, 1e-33)])
def test_stem_weight_gradient_beyond_the_range_of_the_parts(gpu, xscale, dscale):
    """Operands and results at both ends of float32's range: small ones on the parts of 2^24 their value, sums above 2^80 on the float32 MFMAs (every
    product 2^-24, a rounding for each of at most 52272 of them)."""
    rng = np.random.default_rng(43)
    case = CASES[1]
    x, dy = (rng.uniform(0.5, 1, case["x"]) * xscale).astype(np.float32), (rng.uniform(-1, -0.5, _extents(case)) * dscale).astype(np.float32)
    got, want = _call(x, dy, case["k"], case["rs"], case["p"]), _want(x, dy, case["rs"], case["p"])
    assert (np.abs(got - want) <= 3.2e-3 * np.abs(want) + 52272 * 2.0 ** -126).all()
    assert np.linalg.norm(got / want - 1) <= 1e-5 * np.sqrt(want.size)
