"""The convolution of images with few channels from windows in LDS (csrc/kernels/conv_stem.h): rows of 4, 2 and 1 values a load, paddings of
either parity, remainders of channels, rows and pixels, and float32 operands at the ends of the range."""
import ctypes

import numpy as np
import pytest

import jittor_amd as jt
from jittor_amd import _lib as L

pytestmark = pytest.mark.gpu


def _operand(v, dt):
    if dt == "float32":
        return jt.from_storage(v.astype(np.float32), dt), v.astype(np.float32).astype(np.float64)
    if dt == "float16":
        h = v.astype(np.float16)
        return jt.from_storage(h, dt), h.astype(np.float64)
    bits = (v.astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)
    return jt.from_storage(bits, dt), (bits.astype(np.uint32) << 16).view(np.float32).astype(np.float64)


def _call(x, w, ys, p, odt):
    out = jt.from_storage(np.full(ys, 7, L.NP_STORAGE[odt]), odt)
    jt.sync([x, w, out], True)
    tx, tw, ty = (L.tensor(v.raw_ptr(), v.dtype, v.shape) for v in (x, w, out))
    cp = L.ConvParams(*p)
    L.check(L.load().mjt_conv2d_meta(ctypes.byref(tx), ctypes.byref(tw), ctypes.byref(ty), ctypes.byref(cp)))
    assert "_stem_" in L.last_kernel(), L.last_kernel()
    got = L.d2h(out.raw_ptr(), out.shape, L.NP_STORAGE[odt])
    return (got.astype(np.uint32) << 16).view(np.float32).astype(np.float64) if odt == "bfloat16" else got.astype(np.float64)


def _shape(case):
    (n, c, h, w), (r, s), (sh, sw, ph, pw, dh, dw) = case["x"], case["rs"], case["p"]
    return [n, case["k"], (h + 2 * ph - dh * (r - 1) - 1) // sh + 1, (w + 2 * pw - dw * (s - 1) - 1) // sw + 1]


def _want(xf, wf, ys, p):
    sh, sw, ph, pw, dh, dw = p
    (n, k, oh, ow), (r, s) = ys, wf.shape[2:]
    xp = np.pad(xf, ((0, 0), (0, 0), (ph, ph), (pw, pw)))
    y = np.zeros((k, n * oh * ow))
    for i in range(r):
        for j in range(s):
            patch = xp[:, :, i * dh:i * dh + (oh - 1) * sh + 1:sh, j * dw:j * dw + (ow - 1) * sw + 1:sw]
            y += wf[:, :, i, j] @ np.ascontiguousarray(patch.transpose(1, 0, 2, 3)).reshape(xf.shape[1], -1)
    return y.reshape(k, n, oh, ow).transpose(1, 0, 2, 3)


CASES = [
    dict(x=(3, 3, 224, 224), k=64, rs=(7, 7), p=(2, 2, 3, 3, 1, 1)),
    dict(x=(31, 3, 65, 65), k=50, rs=(7, 7), p=(2, 2, 3, 3, 1, 1)),        # odd rows: single values; the last channels and pixels are short
    dict(x=(2, 3, 63, 90), k=20, rs=(7, 7), p=(2, 2, 2, 2, 1, 1)),        # pairs, even padding, one half of the channels
    dict(x=(13, 3, 50, 64), k=70, rs=(7, 7), p=(1, 2, 0, 0, 1, 1)),        # no padding, vertical stride 1, two blocks of channels
    dict(x=(20, 1, 64, 64), k=16, rs=(5, 5), p=(2, 2, 2, 2, 1, 1)),        # one channel: an odd number of rows of taps
    dict(x=(72, 2, 64, 48), k=33, rs=(4, 8), p=(3, 2, 1, 2, 2, 1)),        # eight taps, dilated rows, vertical stride 3
    dict(x=(10, 3, 40, 300), k=64, rs=(7, 7), p=(2, 2, 6, 5, 1, 1)),       # more padding than the taps' half
]


@pytest.mark.parametrize("case", CASES)
def test_stem_convolution(gpu, case):
    """16 bits: products are exact, sums float32 (at most 14 roundings of 16 products: 2e-6 of the sum of magnitudes), one rounding or
    truncation of the result.  float32: what the parts leave out is below 2^-24 of a product, 60 roundings 2^-24 each: 5e-6."""
    rng = np.random.default_rng(31)
    ys = _shape(case)
    for dt in ("float32", "bfloat16", "float16"):
        x, xf = _operand(rng.standard_normal(case["x"]), dt)
        w, wf = _operand(rng.standard_normal((case["k"], case["x"][1], *case["rs"])), dt)
        want, mag = _want(xf, wf, ys, case["p"]), _want(np.abs(xf), np.abs(wf), ys, case["p"])
        for odt in ("float32",) if dt == "float32" else ("float32", dt):
            got = _call(x, w, ys, case["p"], odt)
            bound = 5e-6 * mag + (0 if odt == "float32" else np.abs(want) * (2.0 ** -7 if dt == "bfloat16" else 2.0 ** -10) + 1e-6)
            assert (np.abs(got - want) <= bound).all(), (dt, odt, float(np.abs(got - want).max()))
            if dt == "float32":
                assert np.linalg.norm(got - want) <= 5e-7 * np.linalg.norm(want)


@pytest.mark.parametrize("case", [CASES[i] for i in (1, 2, 4)])
@pytest.mark.parametrize("dt", ["float32", "bfloat16"])
def test_stem_convolution_keeps_infinities_in_their_windows(gpu, case, dt):
    """Positive whole numbers and an infinity in every corner: what sees one is infinite, all else is exact and nothing is NaN."""
    rng = np.random.default_rng(32)
    n, c, h, w_ = case["x"]
    ys = _shape(case)
    v = rng.integers(1, 9, case["x"]).astype(np.float32)
    for i, (a, b) in enumerate([(0, 0), (0, w_ - 1), (h - 1, 0), (h - 1, w_ - 1), (h // 2, w_ // 2)]):
        v[i % n, i % c, a, b] = np.inf
    x, xf = _operand(v, dt)
    w, wf = _operand(rng.integers(1, 9, (case["k"], c, *case["rs"])).astype(np.float32), dt)
    got = _call(x, w, ys, case["p"], "float32")
    seen = _want(np.isinf(xf).astype(float), np.ones_like(wf), ys, case["p"]) > 0
    assert seen.any() and not seen.all()
    assert np.array_equal(np.isinf(got), seen) and not np.isnan(got).any()
    want = _want(np.where(np.isinf(xf), 0, xf), wf, ys, case["p"])
    assert np.array_equal(got[~seen], want[~seen])


@pytest.mark.parametrize("xscale,wscale", [(1e-33, 1e-2), (1e-20, 1e-20), (1e18, 1e18), (1e-2, 1e-33), (1e38, 1e-30)])
def test_stem_convolution_beyond_the_range_of_the_parts(gpu, xscale, wscale):
    """Operands and results at both ends of float32's range: small ones on the parts of 2^24 their value, those above 2^104 and sums above 2^80 on
    the float32 MFMAs, which keep 2^-24 of every product (147 roundings: 1e-5 of the sum of magnitudes)."""
    rng = np.random.default_rng(33)
    case = CASES[1]
    ys = _shape(case)
    x, xf = _operand(rng.uniform(0.5, 1, case["x"]) * xscale, "float32")
    w, wf = _operand(rng.uniform(-1, -0.5, (case["k"], 3, 7, 7)) * wscale, "float32")
    got, want = _call(x, w, ys, case["p"], "float32"), _want(xf, wf, ys, case["p"])
    assert (np.abs(got - want) <= 1e-5 * np.abs(want) + 147 * 2.0 ** -126).all()
