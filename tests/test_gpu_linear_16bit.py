"""The gradients of a 16-bit linear layer are matrix products: dy comes to them through the float32 that the forward sum runs in
(python/jittor/src/opt/tuner/matmul_tuner.cc:16-104 for the pattern, ops/reduce_op.cc:259-266 for the casts)."""
import numpy as np
import pytest

import jittor_amd as jt
from jittor_amd import dtypes, executor


def _var(shape, dtype, rng):
    """A Var of standard normal values of the type, and these values in 64 bits."""
    v = rng.standard_normal(shape).astype(np.float32)
    if dtype == "bfloat16":
        bits = dtypes.f32_to_bf16_bits(v)
        return jt.from_storage(bits, dtype), dtypes.bf16_bits_to_f32(bits).astype(np.float64)
    v = v.astype(dtype)
    return jt.from_storage(v, dtype), v.astype(np.float64)


def _close(got, want, size, terms, dtype):
    """A float32 sum of exact products (size: the sum of their absolute values), narrowed once: bfloat16 keeps the upper 16 bits (2^-7 of
    the value), float16 rounds to nearest (2^-11, 2^-25 below its normal range)."""
    summed = size * (terms + 2) * 2.0 ** -24 * 1.01
    one = (np.abs(want) + summed) * 2.0 ** -7 if dtype == "bfloat16" else (np.abs(want) + summed) * 2.0 ** -11 + 2.0 ** -25
    assert (np.abs(got.astype(np.float64) - want) <= one + summed).all()


# one tile and its edges, sums below and past a stage, rows that are no 16-byte multiples
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("m,k,n", [(2, 16, 16), (2, 64, 3), (17, 33, 65), (64, 64, 64), (129, 128, 127), (300, 72, 520), (1024, 16, 48)])
def test_gradients(gpu, dtype, m, k, n):
    rng = np.random.default_rng(m * 7 + n)
    (x, fx), (w, fw), (g, fg) = (_var(s, dtype, rng) for s in ((m, k), (n, k), (m, n)))
    matched = executor.stats["matmul_matches"]
    with jt.flag_scope(enable_replay=0):
        y = jt.nn.linear(x, w)
        dx, dw = jt.grad((y * g).sum(), [x, w])
        jt.sync([y, dx, dw])
    assert executor.stats["matmul_matches"] - matched == 3
    for got, p, q in ((y, fx, fw.T), (dx, fg, fw), (dw, fg.T, fx)):
        assert got.dtype == dtype
        _close(got.numpy(), p @ q, np.abs(p) @ np.abs(q), p.shape[1], dtype)


def _products(targets):
    """What the matcher makes of the sums among the pending ops: the operands' ids and layouts."""
    units = [executor._match_matmul(op) for op in executor._pending_ops(targets) if type(op).__name__ == "ReduceOp"]
    return [([v.id for v in u.inputs], u.trans) for u in units if u is not None]


@pytest.mark.parametrize("dtype", ["bfloat16", "float16", "float32"])
def test_gradients_are_recognised(compile_only, dtype):
    rng = np.random.default_rng(0)
    x, w, g = (_var(s, dtype, rng)[0] for s in ((5, 7), (3, 7), (5, 3)))
    y = jt.nn.linear(x, w)
    grads = jt.grad((y * g).sum(), [x, w])
    found = _products([y] + grads)
    assert sorted(trans for _, trans in found) == [(False, False), (False, True), (True, False)]
    assert sorted(sorted(ids) for ids, _ in found) == sorted(sorted(ids) for ids in ([x.id, w.id], [g.id, w.id], [g.id, x.id]))


@pytest.mark.parametrize("dtype,through,same", [("bfloat16", "float32", True), ("float16", "float64", True), ("float32", "float64", True),
                                                ("bfloat16", "float16", False), ("float32", "bfloat16", False), ("float32", "int32", False)])
def test_casts_that_change_values_are_kept(compile_only, dtype, through, same):
    """An operand that was narrowed on the way to the product is not the operand: only casts through wider float types are looked
    through."""
    rng = np.random.default_rng(0)
    a, b = _var((4, 6), dtype, rng)[0], _var((6, 5), dtype, rng)[0]
    spread = a.cast(through).broadcast([4, 6, 5], [2]).cast(dtype)
    found = _products([(spread * b.broadcast([4, 6, 5], [0])).sum([1])])
    assert found == ([([a.id, b.id], (False, False))] if same else [])
