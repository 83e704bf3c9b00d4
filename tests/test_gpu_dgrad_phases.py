"""The input gradient of strided convolutions, all phases in one launch (csrc/kernels/conv_dgrad_phases.h): tiles that straddle rows and
images, remainders of channels and maps, strides along one axis, dilation, phases without taps, padding of any kind."""
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


def _call(dy, w, xs, p, odt):
    out = jt.from_storage(np.full(xs, 7, L.NP_STORAGE[odt]), odt)
    jt.sync([out], True)
    td, tw, tx = (L.tensor(v.raw_ptr(), v.dtype, v.shape) for v in (dy, w, out))
    cp = L.ConvParams(*p)
    L.check(L.load().mjt_conv2d_meta_dgrad(ctypes.byref(td), ctypes.byref(tw), ctypes.byref(tx), ctypes.byref(cp)))
    assert "_dgrad_c" in L.last_kernel(), L.last_kernel()
    got = L.d2h(out.raw_ptr(), out.shape, L.NP_STORAGE[odt])
    return (got.astype(np.uint32) << 16).view(np.float32).astype(np.float64) if odt == "bfloat16" else got.astype(np.float64)


def _want(df, wf, hw, p):
    sh, sw, ph, pw, dh, dw = p
    n, k, oh, ow = df.shape
    c, r, s = wf.shape[1:]
    dx = np.zeros((n, c, max(hw[0] + 2 * ph, (oh - 1) * sh + (r - 1) * dh + 1), max(hw[1] + 2 * pw, (ow - 1) * sw + (s - 1) * dw + 1)))
    a = np.ascontiguousarray(df.transpose(0, 2, 3, 1)).reshape(-1, k)
    for i in range(r):
        for j in range(s):
            g = (a @ np.ascontiguousarray(wf[:, :, i, j])).reshape(n, oh, ow, c).transpose(0, 3, 1, 2)
            dx[:, :, i * dh:i * dh + (oh - 1) * sh + 1:sh, j * dw:j * dw + (ow - 1) * sw + 1:sw] += g
    return dx[:, :, ph:ph + hw[0], pw:pw + hw[1]]


CASES = [
    dict(x=(64, 256, 28, 28), k=256, rs=(3, 3), p=(2, 2, 1, 1, 1, 1)),    # tiles of 128 positions, full channels
    dict(x=(2, 70, 28, 28), k=40, rs=(3, 3), p=(2, 2, 1, 1, 1, 1)),       # tiles of 64; the last channels of either kind are short
    dict(x=(5, 64, 27, 27), k=30, rs=(3, 3), p=(2, 2, 1, 1, 1, 1)),       # odd maps: the last phase ends a position early
    dict(x=(9, 33, 13, 7), k=65, rs=(3, 3), p=(2, 2, 1, 1, 1, 1)),        # a tile covers several images; odd rows of dy
    dict(x=(3, 32, 14, 15), k=17, rs=(5, 5), p=(2, 2, 2, 2, 1, 1)),       # shifts to both sides, 25 taps
    dict(x=(4, 48, 14, 14), k=130, rs=(1, 1), p=(2, 2, 0, 0, 1, 1)),      # three phases that no tap reaches; four groups of 16 channels a stage
    dict(x=(4, 48, 9, 14), k=20, rs=(2, 2), p=(2, 2, 0, 0, 1, 1)),        # no overlap, two groups; the last row of dx is not reached
    dict(x=(3, 64, 12, 11), k=64, rs=(3, 3), p=(1, 2, 1, 1, 1, 1)),       # strides along one axis
    dict(x=(3, 64, 11, 12), k=64, rs=(3, 3), p=(2, 1, 1, 1, 1, 1)),
    dict(x=(2, 64, 16, 15), k=64, rs=(3, 3), p=(2, 2, 2, 2, 2, 2)),       # dilation: all taps in one phase
    dict(x=(2, 64, 16, 15), k=33, rs=(3, 2), p=(2, 2, 0, 0, 3, 1)),
    dict(x=(1, 8, 1, 1), k=3, rs=(3, 3), p=(2, 2, 1, 1, 1, 1)),           # a single position
    dict(x=(1, 16, 40, 150), k=16, rs=(3, 7), p=(2, 2, 1, 0, 1, 1)),      # long rows, no padding along them
]


@pytest.mark.parametrize("case", CASES)
def test_strided_input_gradient(gpu, case):
    """Products are exact and sums float32 (at most 256 * 9 terms, 16 products a rounding: 2^-24 * 150, below 1e-5 of the sum of
    magnitudes), and one rounding (or truncation) for a result of 16 bits."""
    rng = np.random.default_rng(21)
    n, c, h, w = case["x"]
    (r, s), p = case["rs"], case["p"]
    sh, sw, ph, pw, dh, dw = p
    oh, ow = (h + 2 * ph - dh * (r - 1) - 1) // sh + 1, (w + 2 * pw - dw * (s - 1) - 1) // sw + 1
    for dt in ("bfloat16", "float16"):
        dy, df = _operand(rng.standard_normal((n, case["k"], oh, ow)), dt)
        wt, wf = _operand(rng.standard_normal((case["k"], c, r, s)), dt)
        jt.sync([dy, wt], True)
        want, mag = _want(df, wf, (h, w), p), _want(np.abs(df), np.abs(wf), (h, w), p)
        for odt in ("float32", dt):
            got = _call(dy, wt, case["x"], p, odt)
            bound = 1e-5 * mag + (0 if odt == "float32" else np.abs(want) * (2.0 ** -7 if dt == "bfloat16" else 2.0 ** -10) + 1e-6)
            assert (np.abs(got - want) <= bound).all(), float(np.abs(got - want).max())


@pytest.mark.parametrize("case", [CASES[i] for i in (1, 2, 3, 7, 9)])
def test_strided_input_gradient_keeps_infinities_in_their_taps(gpu, case):
    """An infinity in dy reaches exactly the positions whose taps see it: positive whole numbers, so no sum cancels and all others are exact."""
    rng = np.random.default_rng(22)
    n, c, h, w = case["x"]
    (r, s), p = case["rs"], case["p"]
    sh, sw, ph, pw, dh, dw = p
    oh, ow = (h + 2 * ph - dh * (r - 1) - 1) // sh + 1, (w + 2 * pw - dw * (s - 1) - 1) // sw + 1
    v = rng.integers(1, 9, (n, case["k"], oh, ow)).astype(np.float32)
    hit = np.zeros((n, 1, oh, ow))
    for i, (y, z) in enumerate([(0, 0), (0, ow - 1), (oh - 1, 0), (oh - 1, ow - 1), (oh // 2, ow // 2)]):
        v[i % n, i % case["k"], y, z] = np.inf
        hit[i % n, 0, y, z] = 1
    dy, df = _operand(v, "bfloat16")
    wt, wf = _operand(rng.integers(1, 9, (case["k"], c, r, s)).astype(np.float32), "bfloat16")
    jt.sync([dy, wt], True)
    got = _call(dy, wt, case["x"], p, "float32")
    seen = np.broadcast_to(_want(hit, np.ones((1, 1, r, s)), (h, w), p) > 0, got.shape)
    assert seen.any() and not seen.all()
    assert np.array_equal(np.isinf(got), seen) and not np.isnan(got).any()
    want = _want(np.where(np.isinf(df), 0, df), wf, (h, w), p)
    assert np.array_equal(got[~seen], want[~seen])
