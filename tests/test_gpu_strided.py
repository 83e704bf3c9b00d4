"""The forward convolution at horizontal stride 2 from windows in LDS (csrc/kernels/conv_strided.h): tiles that straddle rows and images,
channels of any multiple, one row phase or two, dilation, padding of any kind."""
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


def _call(x, w, ys, p, odt):
    out = jt.from_storage(np.full(ys, 7, L.NP_STORAGE[odt]), odt)
    jt.sync([x, w, out], True)
    tx, tw, ty = (L.tensor(v.raw_ptr(), v.dtype, v.shape) for v in (x, w, out))
    cp = L.ConvParams(*p)
    L.check(L.load().mjt_conv2d_meta(ctypes.byref(tx), ctypes.byref(tw), ctypes.byref(ty), ctypes.byref(cp)))
    assert "_strided_" in L.last_kernel(), L.last_kernel()
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
            y += np.ascontiguousarray(wf[:, :, i, j]) @ np.ascontiguousarray(patch.transpose(1, 0, 2, 3)).reshape(xf.shape[1], -1)
    return y.reshape(k, n, oh, ow).transpose(1, 0, 2, 3)


CASES = [
    dict(x=(64, 256, 28, 28), k=256, rs=(3, 3), p=(2, 2, 1, 1, 1, 1)),    # tiles of 128 x 128, full channels
    dict(x=(5, 32, 28, 28), k=192, rs=(3, 3), p=(2, 2, 1, 1, 1, 1)),      # three blocks of channels; the last tile is short
    dict(x=(7, 64, 21, 20), k=64, rs=(3, 3), p=(2, 2, 1, 1, 1, 1)),       # a tile covers two images, odd columns of them
    dict(x=(6, 32, 28, 30), k=64, rs=(5, 5), p=(2, 2, 2, 2, 1, 1)),       # shifts to both sides, 25 taps
    dict(x=(20, 96, 14, 14), k=192, rs=(1, 1), p=(2, 2, 0, 0, 1, 1)),     # one row phase of two, two groups of 16 channels a stage: 96 channels are no multiple of 64
    dict(x=(9, 64, 14, 14), k=32, rs=(1, 1), p=(1, 2, 0, 0, 1, 1)),       # 32 channels; vertical stride 1
    dict(x=(20, 64, 28, 24), k=64, rs=(2, 2), p=(2, 2, 0, 0, 1, 1)),      # two groups; no overlap
    dict(x=(9, 64, 12, 22), k=64, rs=(3, 3), p=(1, 2, 1, 1, 1, 1)),       # vertical stride 1
    dict(x=(9, 64, 26, 26), k=64, rs=(3, 3), p=(2, 2, 2, 2, 2, 2)),       # dilation: all taps in one phase
    dict(x=(9, 32, 26, 24), k=64, rs=(3, 2), p=(2, 2, 0, 5, 3, 1)),       # more padding than taps reach
    dict(x=(2, 32, 40, 60), k=32, rs=(3, 7), p=(2, 2, 1, 0, 1, 1)),       # long rows, no padding along them
]


@pytest.mark.parametrize("case", CASES)
def test_strided_convolution(gpu, case):
    """Products are exact and sums float32 (at most 256 * 9 terms, 16 products a rounding: 2^-24 * 150, below 1e-5 of the sum of
    magnitudes), and one rounding (or truncation) for a result of 16 bits."""
    rng = np.random.default_rng(51)
    ys = _shape(case)
    for dt in ("bfloat16", "float16"):
        x, xf = _operand(rng.standard_normal(case["x"]), dt)
        w, wf = _operand(rng.standard_normal((case["k"], case["x"][1], *case["rs"])), dt)
        want, mag = _want(xf, wf, ys, case["p"]), _want(np.abs(xf), np.abs(wf), ys, case["p"])
        for odt in ("float32", dt):
            got = _call(x, w, ys, case["p"], odt)
            bound = 1e-5 * mag + (0 if odt == "float32" else np.abs(want) * (2.0 ** -7 if dt == "bfloat16" else 2.0 ** -10) + 1e-6)
            assert (np.abs(got - want) <= bound).all(), float(np.abs(got - want).max())


@pytest.mark.parametrize("case", [CASES[i] for i in (1, 2, 3, 5, 7, 8)])
def test_strided_convolution_keeps_infinities_in_their_windows(gpu, case):
    """Positive whole numbers and infinities at the borders: what sees one is infinite, all else is exact and nothing is NaN."""
    rng = np.random.default_rng(52)
    n, c, h, w_ = case["x"]
    ys = _shape(case)
    v = rng.integers(1, 9, case["x"]).astype(np.float32)
    for i, (a, b) in enumerate([(0, 0), (0, w_ - 1), (h - 1, 0), (h - 1, w_ - 1), (h // 2, w_ // 2)]):
        v[i % n, 3 * i % c, a, b] = np.inf
    x, xf = _operand(v, "bfloat16")
    w, wf = _operand(rng.integers(1, 9, (case["k"], c, *case["rs"])).astype(np.float32), "bfloat16")
    got = _call(x, w, ys, case["p"], "float32")
    seen = _want(np.isinf(xf).astype(float), np.ones_like(wf), ys, case["p"]) > 0
    assert not seen.all()
    assert np.array_equal(np.isinf(got), seen) and not np.isnan(got).any()
    want = _want(np.where(np.isinf(xf), 0, xf), wf, ys, case["p"])
    assert np.array_equal(got[~seen], want[~seen])
