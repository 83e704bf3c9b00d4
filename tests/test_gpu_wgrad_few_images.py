"""Weight gradients of small 16-bit maps whose images make no chunks (or are fewer than six) take the product that gathers its operands:
against 64 bits (python/jittor/nn.py:1251-1262 differentiated; opt/tuner/conv_tuner.cc:375-397)."""
import numpy as np
import pytest

import jittor_amd as jt
from jittor_amd import dtypes, executor

pytestmark = pytest.mark.gpu


def _var(shape, dtype, rng):
    v = rng.standard_normal(shape).astype(np.float32)
    if dtype == "bfloat16":
        bits = dtypes.f32_to_bf16_bits(v)
        return jt.from_storage(bits, dtype), dtypes.bf16_bits_to_f32(bits).astype(np.float64)
    return jt.from_storage(v.astype(dtype), dtype), v.astype(dtype).astype(np.float64)


# one image, odd numbers of them, odd and even planes, extents of one, channels that are no multiples of a tile; 1x1, strides
@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("shape,k,r,stride", [((1, 64, 14, 14), 32, 3, 1), ((1, 130, 14, 14), 66, 1, 1), ((3, 48, 7, 7), 40, 3, 1), ((5, 17, 11, 9), 33, 3, 2), ((4, 32, 14, 14), 64, 3, 1),
                                              ((2, 300, 13, 13), 20, 3, 1), ((1, 16, 1, 3), 8, 3, 1), ((51, 16, 11, 11), 24, 5, 1), ((2, 256, 14, 14), 256, 1, 1)])
def test_weight_gradient(gpu, dtype, shape, k, r, stride):
    rng = np.random.default_rng(shape[0] * shape[1])
    n, c, h, w = shape
    p = r // 2
    oh, ow = ((e + 2 * p - r) // stride + 1 for e in (h, w))
    x, fx = _var(shape, dtype, rng)
    wt, _ = _var((k, c, r, r), dtype, rng)
    g, fg = _var((n, k, oh, ow), dtype, rng)
    before = executor.stats["wgrad_chunked"]
    dw, = jt.grad((jt.nn.conv2d(x, wt, stride=stride, padding=p) * g).sum(), [wt])
    dw.sync()
    assert dw.dtype == dtype and executor.stats["wgrad_chunked"] == before
    got = dw.numpy().astype(np.float64)
    fx = np.pad(fx, ((0, 0), (0, 0), (p, p), (p, p)))
    d = fg.transpose(1, 0, 2, 3).reshape(k, -1)
    for i in range(r):
        for j in range(r):
            t = fx[:, :, i:i + (oh - 1) * stride + 1:stride, j:j + (ow - 1) * stride + 1:stride].transpose(0, 2, 3, 1).reshape(-1, c)
            want, size = d @ t, np.abs(d) @ np.abs(t)
            # a float32 sum of exact products in any order, narrowed once
            bound = size * (n * oh * ow + 2) * 2.0 ** -24 * 1.01
            bound = bound + (np.abs(want) + bound) * (2.0 ** -7 if dtype == "bfloat16" else 2.0 ** -11) + (0 if dtype == "bfloat16" else 2.0 ** -25)
            assert (np.abs(got[:, :, i, j] - want) <= bound).all()
