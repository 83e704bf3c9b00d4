"""Input gradients of small strided convolutions in one launch (kernels/conv_dgrad_direct.h), against 64 bits, with a group behind them and with
weights that are not finite."""
import ctypes

import numpy as np
import pytest

import jittor_amd as jt
from jittor_amd import _lib as L, dtypes

pytestmark = pytest.mark.gpu


def _var(v, dtype):
    if dtype == "bfloat16":
        bits = dtypes.f32_to_bf16_bits(v)
        return jt.from_storage(bits, dtype), dtypes.bf16_bits_to_f32(bits).astype(np.float64)
    v = v.astype(dtype)
    return jt.from_storage(v, dtype), v.astype(np.float64)


def _reference(dy, w, shape, s, p, absolute=False):
    n, c, h, x = shape
    out = np.zeros((n, c, h + 2 * p, x + 2 * p))
    for i in range(w.shape[2]):
        for j in range(w.shape[3]):
            with np.errstate(invalid="ignore"):
                t = np.einsum("nkhx,kc->nchx", dy, w[:, :, i, j])
            out[:, :, i:i + (dy.shape[2] - 1) * s[0] + 1:s[0], j:j + (dy.shape[3] - 1) * s[1] + 1:s[1]] += t
    return out[:, :, p:p + h, p:p + x]


# lanes that share a result: one, four, eight, sixteen; channels that are no multiple of them; windows smaller and larger than the stride; the last
# workgroup part filled; 16 bits where no kernel of all phases is (stride 3)
@pytest.mark.parametrize("dtype,shape,k,r,s", [("float32", (1, 1, 2, 2), 1, 3, 2), ("float32", (4, 16, 6, 6), 16, 3, 2), ("float32", (2, 5, 8, 12), 3, 1, 2), ("float32", (3, 7, 10, 6), 33, 5, 2),
                                               ("float32", (1, 4, 9, 9), 9, 3, 3), ("float32", (2, 3, 8, 8), 4, 2, 4), ("bfloat16", (2, 6, 9, 12), 10, 3, 3), ("float16", (1, 9, 6, 6), 40, 5, 3)])
def test_input_gradient(gpu, dtype, shape, k, r, s):
    rng = np.random.default_rng(k + r)
    n, c, h, x = shape
    p = r // 2 if (h + 2 * (r // 2) - r) // s + 1 >= h // s else 0
    oh, ow = ((e + 2 * p - r) // s + 1 for e in (h, x))
    dy, fy = _var(rng.standard_normal((n, k, oh, ow)).astype(np.float32), dtype)
    w, fw = _var(rng.standard_normal((k, c, r, r)).astype(np.float32), dtype)
    dx = jt.zeros(list(shape), dtype)
    td, tw, tx = (L.tensor(v.raw_ptr(), dtype, v.shape) for v in (dy, w, dx))
    L.check(L.load().mjt_conv2d_meta_dgrad(ctypes.byref(td), ctypes.byref(tw), ctypes.byref(tx), ctypes.byref(L.ConvParams(s, s, p, p, 1, 1))))
    assert "mjt_conv_direct_dgrad" in L.last_kernel(), L.last_kernel()
    got = L.d2h(dx.raw_ptr(), dx.shape, L.NP_STORAGE[dtype])
    got = (dtypes.bf16_bits_to_f32(got) if dtype == "bfloat16" else got).astype(np.float64)
    want, size = _reference(fy, fw, shape, (s, s), p), _reference(np.abs(fy), np.abs(fw), shape, (s, s), p)
    bound = size * (k * r * r + 6) * 2.0 ** -24                             # a float32 sum of at most k r r products, some lanes' parts added up
    bound = bound + (np.abs(want) + bound) * {"float32": 0, "bfloat16": 2.0 ** -7, "float16": 2.0 ** -11}[dtype] + 2.0 ** -25 * (dtype == "float16")
    assert (np.abs(got - want) <= bound).all()


def test_group_behind_and_infinite_weights(gpu):
    """The mask of a relu behind the gradient gives the same bits as by itself; an infinite weight stays with the results that its tap
    reaches."""
    rng = np.random.default_rng(0)
    x = jt.array(rng.standard_normal((3, 8, 6, 6)).astype(np.float32))
    v = rng.standard_normal((16, 8, 3, 3)).astype(np.float32)
    v[3, 5, 0, 2] = np.inf
    w, g = jt.array(v), jt.array(rng.standard_normal((3, 16, 3, 3)).astype(np.float32))
    out = []
    for fused in (1, 0):
        with jt.flag_scope(enable_product_fusion=fused):
            for _ in range(3):
                h = jt.nn.relu(x)
                dx, = jt.grad((jt.nn.conv2d(h, w, stride=2, padding=1) * g).sum(), [x])
                jt.sync([dx, h])
                out.append(dx.numpy())
    for o in out[1:]:
        assert np.array_equal(o, out[0], equal_nan=True)
    want = _reference(g.numpy().astype(np.float64), v.astype(np.float64), (3, 8, 6, 6), (2, 2), 1)
    mask = x.numpy() > 0
    assert np.array_equal(np.isfinite(out[0][mask]), np.isfinite(want[mask])) and (~np.isfinite(want)).sum() < want.size // 8
