"""Convolutions of few tiles and long sums: the sum in slices (kernels/gemm_mfma.h with CONV and SLICED), against the convolution in 64 bits."""
import numpy as np
import pytest

import jittor_amd as jt
from jittor_amd import _lib, dtypes

pytestmark = pytest.mark.gpu


def _var(v, dtype):
    """A Var of the values rounded to the type, and what they are then in 64 bits."""
    if dtype == "bfloat16":
        bits = dtypes.f32_to_bf16_bits(v)
        return jt.from_storage(bits, dtype), dtypes.bf16_bits_to_f32(bits).astype(np.float64)
    v = v.astype(dtype)
    return jt.from_storage(v, dtype), v.astype(np.float64)


def _conv(x, w, stride):
    r, (oh, ow) = w.shape[2], [(e + 2 * (w.shape[2] // 2) - w.shape[2]) // stride + 1 for e in x.shape[2:]]
    x = np.pad(x, ((0, 0), (0, 0), (r // 2, r // 2), (r // 2, r // 2)))
    y = 0.0
    with np.errstate(invalid="ignore"):
        for i in range(r):
            for j in range(r):
                tap = x[:, :, i:i + (oh - 1) * stride + 1:stride, j:j + (ow - 1) * stride + 1:stride]
                y = y + np.matmul(w[:, :, i, j], tap.reshape(x.shape[0], x.shape[1], -1)).reshape(x.shape[0], -1, oh, ow)
    return y


def _check(shape, k, r, stride, dtype, seed=0, values=None):
    rng = np.random.default_rng(seed)
    n, c, h, w = shape
    x, fx = _var(rng.standard_normal(shape).astype(np.float32) if values is None else values, dtype)
    wt, fw = _var(rng.standard_normal((k, c, r, r)).astype(np.float32), dtype)
    with jt.flag_scope(enable_replay=0):
        y = jt.nn.conv2d(x, wt, stride=stride, padding=r // 2)
        got = y.numpy().astype(np.float64)
    name = _lib.load().mjt_last_kernel().decode()
    want, size = _conv(fx, fw, stride), _conv(np.abs(fx), np.abs(fw), stride)
    # a float32 sum of c r r terms in any order, cut into up to 16 slices, its terms exact (16 bits) or to 2^-24; then one narrowing
    bound = size * (c * r * r + 18) * 2.0 ** -24 * 1.01
    if dtype == "bfloat16":
        bound = bound + (np.abs(want) + bound) * 2.0 ** -7
    elif dtype == "float16":
        bound = bound + (np.abs(want) + bound) * 2.0 ** -11 + 2.0 ** -25
    finite = np.isfinite(want)
    assert (np.abs(got - want)[finite] <= bound[finite]).all()
    assert np.array_equal(got[~finite], want[~finite], equal_nan=True)
    return name


# tiles and their edges, sums that end inside a stage and whose last slice is short, rows of weights that are no 16-byte multiples, 1x1
@pytest.mark.parametrize("dtype", ["float32", "bfloat16", "float16"])
@pytest.mark.parametrize("shape,k,r,stride", [((1, 215, 7, 7), 17, 3, 1), ((3, 67, 9, 5), 65, 3, 2), ((2, 300, 5, 5), 64, 5, 1), ((5, 768, 7, 7), 130, 1, 1),
                                              ((1, 512, 1, 3), 3, 3, 1), ((4, 160, 13, 13), 64, 3, 1), ((1, 1024, 5, 4), 64, 1, 1), ((3, 1024, 14, 14), 256, 1, 1)])
def test_long_sums(gpu, shape, k, r, stride, dtype):
    name = _check(shape, k, r, stride, dtype)
    assert "slices" in name or (dtype != "float32" and shape[3] % 2 == 0)          # (even rows of 16-bit values have kernels of their own)


# any number of slices down to one stage each, of every tile and of sums of few stages
@pytest.mark.parametrize("slices", [2, 3, 5, 16])
@pytest.mark.parametrize("shape,k,r,dtype", [((2, 16, 9, 9), 20, 3, "float32"), ((20, 64, 14, 14), 128, 3, "float32"), ((70, 64, 28, 28), 256, 3, "float32"),
                                             ((9, 30, 11, 11), 70, 3, "bfloat16"), ((64, 24, 27, 27), 160, 3, "float16")])
def test_forced_slices(gpu, monkeypatch, shape, k, r, dtype, slices):
    monkeypatch.setenv("MJT_CONV_SLICES", str(slices))
    assert "slices" in _check(shape, k, r, 1, dtype)


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 3e38])
def test_values_beyond_the_parts_range(gpu, value):
    """A slice whose sums of bfloat16 parts are not finite is summed again by the float32 MFMAs; the others are not."""
    v = np.random.default_rng(1).standard_normal((3, 256, 14, 14)).astype(np.float32) * 1e-3
    v[1, 200, 5, 6] = value
    v[2, 3, 0, 13] = 1e-40
    with np.errstate(invalid="ignore", over="ignore"):
        if abs(value) == 3e38:
            v[1, 200, 5, 6] = 3e37
        assert "slices" in _check((3, 256, 14, 14), 256, 3, 1, "float32", values=v)


@pytest.mark.parametrize("dtype,shape,k", [("float32", (2, 256, 7, 7), 64), ("float32", (1, 130, 5, 3), 3), ("bfloat16", (3, 270, 9, 9), 70), ("float16", (1, 200, 7, 5), 18)])
def test_group_behind(gpu, dtype, shape, k):
    """A group behind a sliced convolution runs where the slices are added up, on the same values as by itself."""
    rng = np.random.default_rng(2)
    x, _ = _var(rng.standard_normal(shape).astype(np.float32), dtype)
    w, _ = _var(rng.standard_normal((k, shape[1], 3, 3)).astype(np.float32), dtype)
    b, _ = _var(rng.standard_normal((1, k, 1, 1)).astype(np.float32), dtype)
    out = {}
    for fused in (1, 0):
        with jt.flag_scope(enable_product_fusion=fused):
            for _ in range(4):                                 # executed, replayed by its calls, recorded, by the recording
                y = jt.nn.conv2d(x, w, padding=1)
                z = jt.nn.relu(y + b)
                only = jt.nn.relu(jt.nn.conv2d(x, w, padding=1) + b)
                jt.sync([y, z])
                got = [v.raw().copy() for v in (y, z, only)]
                for a, c in zip(out.setdefault(0, got), got):
                    assert np.array_equal(a.view(np.uint8), c.view(np.uint8))
