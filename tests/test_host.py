"""Host-side logic without a GPU: the C-ABI library loads and exports every
symbol include/mjt.h declares, descriptors are validated, index expressions
parse as the reference's language, the front end reproduces the constructor
rewrites / dtype rules, and kernels specialise + compile for gfx950."""
import ctypes
import json
import os
import re
import subprocess
import sys
import time

import numpy as np
import pytest

import jittor_amd as jt
import rows_graphs
from jittor_amd import _lib as L

G = json.load(open(os.path.join(os.path.dirname(__file__), "golden", "vectors.json")))
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
P = 0x100000     # fake, aligned device pointer: nothing is launched in compile-only mode


def test_library_exports_every_declared_symbol():
    lib = L.load()
    header = open(os.path.join(ROOT, "include", "mjt.h")).read()
    declared = set(re.findall(r"\b(mjt_[a-z0-9_]+)\s*\(", header))
    assert declared == set(L.EXPORTS), declared ^ set(L.EXPORTS)
    for name in declared:
        assert hasattr(lib, name), name


def test_names_and_codes():
    lib = L.load()
    for i, n in enumerate(L.DTYPES):
        assert lib.mjt_dtype_name(i).decode() == n
    for i, n in enumerate(L.OPS):
        assert lib.mjt_op_name(i).decode() == n
    assert lib.mjt_op_from_name(b"add") == L.OP_CODE["add"]
    assert lib.mjt_op_from_name(b"nope") < 0
    assert lib.mjt_dtype_from_name(b"bfloat16") == L.DTYPE_CODE["bfloat16"]


def test_calls_fail_cleanly_without_init():
    L.shutdown()
    lib = L.load()
    x = L.tensor(P, "float32", [4])
    assert lib.mjt_reduce(ctypes.byref(x), ctypes.byref(x), 3, 1) == -5
    assert b"mjt_init" in lib.mjt_last_error()


def test_expr_affine_and_errors():
    assert L.expr_affine("i3*2-1+i5*3", (4, 5, 6, 7), (1, 2, 3, 4, 5, 6)) == (-1, [0, 0, 0, 2, 0, 3, 0, 0, 0, 0])
    assert L.expr_affine("xshape0-1-i0", (4,), (4,)) == (3, [-1] + [0] * 9)
    assert L.expr_affine("(i1-i3)/2", (4, 4), (4, 4, 4, 4)) is None
    assert L.expr_affine("7/2*i0 + (0-7)/2", (4,), (4,)) == (-3, [3] + [0] * 9)   # C division truncates
    assert L.expr_affine("0x10 + 0b11", (4,), (4,)) == (19, [0] * 10)
    assert L.expr_affine("@e0(i0)", (4,), (4,)) is None
    with pytest.raises(L.MjtError):
        L.expr_affine("i0 // 2", (4,), (4,))
    with pytest.raises(L.MjtError):
        L.expr_affine("i0 +", (4,), (4,))


def test_descriptor_validation(compile_only):
    lib = compile_only.load()
    e = L.c_strings([])
    x, y = L.tensor(P, "float32", [10, 10]), L.tensor(P, "float32", [8, 8])
    # number of indexes must equal x rank (ops/reindex_op.cc:83)
    assert lib.mjt_reindex(ctypes.byref(x), ctypes.byref(y), 1, L.c_strings(["i0"]), 0.0, 0, e, 0, None) == -1
    # '//' is rejected (opt/pass/loop_var_analyze_pass.cc:298-309)
    ex = (L.Tensor * 1)(L.tensor(P, "int32", [1]))
    assert lib.mjt_reindex(ctypes.byref(x), ctypes.byref(y), 2, L.c_strings(["@e0(0) // 1", "@e0(0)"]), 0.0, 0, e, 1, ex) == -1
    # unknown identifier, @eK arity, missing extra
    assert lib.mjt_reindex(ctypes.byref(x), ctypes.byref(y), 2, L.c_strings(["i5", "i0"]), 0.0, 0, e, 0, None) == -1
    assert lib.mjt_reindex(ctypes.byref(x), ctypes.byref(y), 2, L.c_strings(["@e0(i0,i1)", "i0"]), 0.0, 0, e, 1, ex) == -1
    assert lib.mjt_reindex(ctypes.byref(x), ctypes.byref(y), 2, L.c_strings(["@e1(0)", "i0"]), 0.0, 0, e, 1, ex) == -1
    # reindex_reduce: op must be binary and not mean; indexes == rank of the output
    v, o = L.tensor(P, "float32", [3]), L.tensor(P, "float32", [3])
    assert lib.mjt_reindex_reduce(ctypes.byref(v), ctypes.byref(o), L.OP_CODE["mean"], 1, L.c_strings(["i0"]), 0, e, 0, None) == -1
    assert lib.mjt_reindex_reduce(ctypes.byref(v), ctypes.byref(o), L.OP_CODE["exp"], 1, L.c_strings(["i0"]), 0, e, 0, None) == -1
    assert lib.mjt_reindex_reduce(ctypes.byref(v), ctypes.byref(o), L.OP_CODE["add"], 2, L.c_strings(["i0", "i0"]), 0, e, 0, None) == -1
    # reduce: mask must fit, element counts must agree, op must be associative
    big, small = L.tensor(P, "float32", [4, 5]), L.tensor(P, "float32", [4])
    assert lib.mjt_reduce(ctypes.byref(big), ctypes.byref(small), L.OP_CODE["add"], 0b100) == -1
    assert lib.mjt_reduce(ctypes.byref(big), ctypes.byref(small), L.OP_CODE["add"], 0b01) == -1
    assert lib.mjt_reduce(ctypes.byref(big), ctypes.byref(small), L.OP_CODE["subtract"], 0b10) == -1
    assert lib.mjt_reduce(ctypes.byref(big), ctypes.byref(small), L.OP_CODE["add"], 0b10) == 0


def _fused(lib, shape, vars_, ops_):
    va = (L.FusedVar * len(vars_))()
    for i, (role, dt_, mask) in enumerate(vars_):
        va[i].role, va[i].dtype, va[i].ptr, va[i].bcast_mask = role, L.DTYPE_CODE[dt_], P, mask
    oa = (L.FusedOp * len(ops_))()
    for i, (kind, op, ins, out) in enumerate(ops_):
        oa[i].kind, oa[i].op, oa[i].out = kind, L.OP_CODE[op] if op else 0, out
        for j, v in enumerate(ins):
            oa[i].inp[j] = v
    d = L.FusedDesc()
    d.ndim = len(shape)
    for i, s in enumerate(shape):
        d.shape[i] = s
    d.n_vars, d.vars, d.n_ops, d.ops = len(vars_), va, len(ops_), oa
    return lib.mjt_fused_elementwise(ctypes.byref(d))


def test_kernels_specialise_for_gfx950(compile_only):
    """Compile-only mode builds the same kernels a GPU run would launch."""
    lib = compile_only.load()
    e = L.c_strings([])
    before = L.jit_stats()[0]
    os.environ["MJT_NO_DISK_CACHE"] = "1"
    try:
        # the five benchmark shapes
        x, y = L.tensor(P, "float32", [8192, 4096]), L.tensor(P, "float32", [8192])
        assert lib.mjt_reduce(ctypes.byref(x), ctypes.byref(y), L.OP_CODE["add"], 0b10) == 0, lib.mjt_last_error()
        assert L.last_kernel().startswith("mjt_reduce_row_add")
        x, y = L.tensor(P, "float32", [32, 64, 56, 56]), L.tensor(P, "float32", [32, 64, 56, 56, 3, 3])
        assert lib.mjt_reindex(ctypes.byref(x), ctypes.byref(y), 4, L.c_strings(["i0", "i1", "i2+i4-1", "i3+i5-1"]),
                               0.0, 0, e, 0, None) == 0, lib.mjt_last_error()
        assert L.last_kernel().startswith("mjt_window_gather")
        v, o = L.tensor(P, "float32", [1 << 24]), L.tensor(P, "float32", [1 << 20])
        ex = (L.Tensor * 1)(L.tensor(P, "int32", [1 << 24]))
        for op in ("add", "maximum"):
            assert lib.mjt_reindex_reduce(ctypes.byref(v), ctypes.byref(o), L.OP_CODE[op], 1, L.c_strings(["@e0(i0)"]),
                                          0, e, 1, ex) == 0, lib.mjt_last_error()
            assert L.last_kernel().startswith("mjt_scatter1d_" + op)
        vars_ = [(0, "float32", 0), (0, "float32", 0b101), (0, "float32", 0b011), (3, "float32", 0),
                 (1, "float32", 0), (1, "float32", 0), (1, "bool", 0), (1, "float32", 0), (1, "float32", 0),
                 (1, "float32", 0), (1, "float32", 0), (2, "float32", 0)]
        ops_ = [(1, "multiply", [0, 1], 4), (1, "add", [4, 2], 5), (1, "greater", [5, 3], 6), (2, None, [6, 5, 3], 7),
                (0, "negative", [7], 8), (0, "exp", [8], 9), (0, "sigmoid", [0], 10), (1, "multiply", [9, 10], 11)]
        assert _fused(lib, [64, 512, 1024], vars_, ops_) == 0, lib.mjt_last_error()
        # a generic gather with extras and a generic scatter
        x, y = L.tensor(P, "float32", [10, 10]), L.tensor(P, "float32", [8, 8])
        ex2 = (L.Tensor * 2)(L.tensor(P, "int32", [1]), L.tensor(P, "float32", [10, 10]))
        assert lib.mjt_reindex(ctypes.byref(x), ctypes.byref(y), 2, L.c_strings(["@e0(0)", "@e1(0,i0 / @e0(0))"]),
                               0.0, 0, e, 2, ex2) == 0, lib.mjt_last_error()
        yy, xx = L.tensor(P, "int16", [3, 10, 10, 4]), L.tensor(P, "int16", [3, 4, 4, 4])
        assert lib.mjt_reindex_reduce(ctypes.byref(yy), ctypes.byref(xx), L.OP_CODE["multiply"], 4,
                                      L.c_strings(["i0", "i1/3", "i2/3", "i3"]), 0, e, 0, None) == 0, lib.mjt_last_error()
    finally:
        del os.environ["MJT_NO_DISK_CACHE"]
    assert L.jit_stats()[0] >= before + 7


def test_fused_graph_validation(compile_only):
    lib = compile_only.load()
    # op reads a var that is produced later
    assert _fused(lib, [8], [(0, "float32", 0), (1, "float32", 0), (2, "float32", 0)],
                  [(0, "exp", [1], 2), (0, "exp", [0], 1)]) == -1
    # output never produced
    assert _fused(lib, [8], [(0, "float32", 0), (2, "float32", 0), (2, "float32", 0)], [(0, "exp", [0], 1)]) == -1
    # binary op code in a unary slot
    assert _fused(lib, [8], [(0, "float32", 0), (2, "float32", 0)], [(0, "add", [0], 1)]) == -1


# ---- front end: constructor rewrites, shapes, dtypes, errors ---------------------------
def _count_ops(v, kind):
    seen, stack, n = set(), [v], 0
    while stack:
        u = stack.pop()
        if u._op is None or u._op.id in seen:
            continue
        seen.add(u._op.id)
        n += u._op.kind == kind
        stack.extend(u._op.inputs)
    return n


def test_binary_inserts_broadcasts_like_the_reference():
    # test/test_broadcast_to_op.py:64-101: 0, 1 or 2 broadcast ops
    a = jt.array([1, 2, 3])
    assert _count_ops(a + 1, "broadcast") == 1
    assert _count_ops(a + a, "broadcast") == 0
    x, y = jt.zeros([3, 1]), jt.zeros([1, 4])
    z = x + y
    assert z.shape == [3, 4] and _count_ops(z, "broadcast") == 2
    assert (jt.zeros([5, 4]) + jt.zeros([4])).shape == [5, 4]
    with pytest.raises(ValueError):
        jt.zeros([3, 4]) + jt.zeros([3, 5])


def test_broadcast_shapes_and_forwarding():
    a = jt.array([1, 2])
    assert a.broadcast([2, 2], [-1]).shape == [2, 2]
    assert a.broadcast([2]) is a                              # forward(x): nothing to broadcast
    assert jt.zeros([512, 1]).broadcast([64, 512, 1024])._op.bcast_mask == 0b101
    assert jt.zeros([1, 1024]).broadcast([64, 512, 1024])._op.bcast_mask == 0b011
    w = jt.zeros([256, 256, 3, 3]).broadcast([64, 256, 256, 56, 56, 3, 3], [0, 3, 4])
    assert w.shape == [64, 256, 256, 56, 56, 3, 3] and w._op.bcast_mask == 0b0011001
    with pytest.raises(ValueError):
        a.broadcast([2, 2], [5])


def test_reduce_shapes_rewrites_and_errors():
    a = jt.array([[1, 2], [3, 4]])
    assert a.sum(-1).shape == [2] and a.sum(-1)._op.reduce_mask == 0b10
    assert a.sum(-2)._op.reduce_mask == 0b01
    assert a.sum().shape == [1] and a.sum().is_scalar
    assert a.sum(1, keepdims=True).shape == [2, 1]
    assert jt.zeros([2, 3, 4, 5]).sum([1, 3]).shape == [2, 4]
    with pytest.raises(ValueError):
        jt.reduce_add(jt.array([1, 2, 3]), 2)                 # test/test_reduce_op.py:50
    h = jt.zeros([4, 4]).bfloat16().sum(1)                    # cast -> reduce(float32) -> cast
    assert h.dtype == "bfloat16" and h._op.kind == "unary" and h._op.inputs[0].dtype == "float32"
    assert jt.array([True, False]).sum().dtype == "int32"
    assert len([n for n in dir(jt) if n.startswith("reduce_")]) >= 10


def test_dtype_rules_of_the_front_end():
    for op, x, y, xs, ys, want in G["dtype_table"]["rows"]:
        assert jt.dtypes.binary_dtype_infer(op, x, y, xs, ys) == want
    a = jt.array([1.0, 2.0, 3.0]).bfloat16()
    assert (a * 1).dtype == "bfloat16"                        # test/test_bf16.py:275-281
    assert (a * jt.array([1.0, 2.0, 3.0])).dtype == "float32"
    assert (a * jt.array([1.0, 2.0, 3.0]).sum()).dtype == "bfloat16"
    assert jt.array([0, 1, 0]).ternary(a, jt.array(1.0)).dtype == "bfloat16"
    assert (a ** a).dtype == "float32"
    i = jt.array([1, 2, 3])
    assert i.dtype == "int32" and jt.array([1.5]).dtype == "float32" and jt.array(np.arange(4, dtype=np.uint8)).dtype == "uint8"
    assert (i / 2).dtype == "float32" and (i // 2).dtype == "int32" and (i < 2).dtype == "bool"
    assert i.sqrt().dtype == "float32" and i.float16().exp().dtype == "float32" and i.float32().round_int().dtype == "int32"
    assert (i.float64() + 1).dtype == "float64"
    assert i.int32() is i                                      # unary_op.cc:867-870 forwards


def test_amp_reg_controls_dtype_inference():
    """The mixed-precision register (nano_string.h:199-277, var.cc:65-71), with the cases the reference checks
    in test/test_fp16.py:208-300: reduce keeps 16 bit only with keep_reduce, white-list ops only with
    keep_white, prefer16 / prefer32 steer float results unless an operand is a scalar, array-like ops follow
    with array_prefer, and conv2d builds its sum under amp_reg | 36 (nn.py:1250)."""
    a = jt.array(np.ones((3, 4), np.float32)).float16()
    assert jt.flags.amp_reg == 0
    for reg in (0, 1, 2):
        with jt.flag_scope(amp_reg=reg):
            assert a.maximum(a).max().dtype == "float32"                  # reduce_dtype_infer
            assert (a ** a).dtype == "float32"                            # white list
    with jt.flag_scope(amp_reg=2 + 4):
        assert a.sum().dtype == "float16" and a.max().dtype == "float16"  # test_fp16.py:248-252
    with jt.flag_scope(amp_reg=4):
        s = a.sum()
        assert s.dtype == "float16" and s._op.kind == "unary"             # still cast -> reduce(float32) -> cast
        assert a.max().dtype == "float16" and a.max()._op.kind == "reduce"
    with jt.flag_scope(amp_reg=4 + 32):
        s = a.sum()
        assert s.dtype == "float16" and s._op.kind == "reduce" and s._op.amp == 36
    with jt.flag_scope(amp_reg=2 + 8):
        assert (a ** a).dtype == "float16" and a.exp().dtype == "float16"
    with jt.flag_scope(amp_reg=1):
        assert a.sqrt().dtype == "float32" and (a + a).dtype == "float32"
        assert (a * 2.0).dtype == "float16"                               # a scalar operand does not count
    f = jt.array(np.ones((3, 4), np.float32))
    with jt.flag_scope(amp_reg=2):
        assert (f + f).dtype == "float16" and f.sqrt().dtype == "float16"
    assert jt.array([1.0, 2.0]).dtype == "float32"
    with jt.flag_scope(amp_reg=2 + 16):
        assert jt.array([1.0, 2.0]).dtype == "float16" and jt.array([1.0]).dtype == "float32"
    with jt.flag_scope(amp_level=3):                                      # test_fp16.py:293-299
        assert jt.flags.amp_reg == 12
        assert a.sum().dtype == "float16" and a.mean().dtype == "float16"
        assert a.log().dtype == "float16" and a.exp().dtype == "float16"
    assert jt.flags.amp_reg == 0 and jt.flags.auto_mixed_precision_level == 0
    # conv2d: 16-bit operands give a 16-bit sum without casts; the gradient inherits the register
    x, w = jt.zeros([2, 3, 8, 8]).bfloat16(), jt.zeros([4, 3, 3, 3]).bfloat16()
    y = jt.nn.conv2d(x, w, padding=1)
    assert y.dtype == "bfloat16" and y._op.kind == "reduce" and y._op.amp & 36 == 36
    gw = jt.grad(y.sum(), w)
    assert gw.dtype == "bfloat16" and gw._op.kind == "reduce" and gw._op.reduce_mask == 0b0011001
    assert jt.flags.amp_reg == 0
    with pytest.raises(KeyError):
        jt.flags["no_such_flag"] = 1


def test_reindex_constructor_checks():
    x = jt.zeros([10, 10])
    with pytest.raises(ValueError):
        x.reindex([8, 8], ["i0"])
    y = x.reindex_var([jt.zeros([4, 5]).int32(), jt.zeros([4, 5]).int32()])
    assert y.shape == [4, 5] and y._op.indexes == ["@e0(i0,i1)", "@e1(i0,i1)"]
    v = jt.zeros([3])
    v.reindex_reduce("add", [3], ["i0"])
    for bad in (lambda: v.reindex_reduce("add", [3], []), lambda: v.reindex_reduce("add", [3], ["i0", "i0"]),
                lambda: v.reindex_reduce("???", [3], ["i0"]), lambda: v.reindex_reduce("add", [-1], ["i0"])):
        with pytest.raises(ValueError):
            bad()                                              # test/test_reindex_reduce_op.py:92-97


def test_conv2d_builds_the_meta_op_group():
    x, w = jt.zeros([2, 3, 8, 8]), jt.zeros([4, 3, 3, 3])
    y = jt.nn.conv2d(x, w, padding=1)
    assert y.shape == [2, 4, 8, 8] and y._op.kind == "reduce" and y._op.reduce_mask == 0b1100100
    mul = y._op.inputs[0]._op
    assert mul.kind == "binary" and {i._op.kind for i in mul.inputs} == {"reindex", "broadcast"}
    r = [i for i in mul.inputs if i._op.kind == "reindex"][0]._op
    assert r.indexes == ["i0", "i2", "i3*1-1+i5*1", "i4*1-1+i6*1"]
    assert jt.nn.conv2d(x, w, stride=2, padding=1).shape == [2, 4, 4, 4]


# ---- gradients: graph construction (no execution) -------------------------------------------
def test_grad_graph_is_built_from_path_ops():
    """The gradient of a meta-op is again a meta-op of the path
    (reindex_op.cc:76-80, reindex_reduce_op.cc:45-63, reduce_op.cc:339-362,
    broadcast_to_op.cc:112-117)."""
    import jittor_amd as jt
    from jittor_amd import core
    x = jt.array(np.zeros((2, 3, 8, 8), np.float32))
    xx = x.reindex([2, 3, 4, 4, 2, 2], ["i0", "i1", "i2*2+i4", "i3*2+i5"], overflow_conditions=["i2<0"])
    g = jt.grad(xx.sum(), x)
    assert isinstance(g._op, core.ReindexReduceOp) and g._op.op == "add" and g.shape == x.shape
    assert g._op.indexes == xx._history[0].indexes and g._op.overflow_conditions == ["i2<0"]
    y = x.reindex_reduce("add", [2, 3, 4, 4], ["i0", "i1", "i2/2", "i3/2"])
    g = jt.grad(y.sum(), x)
    assert isinstance(g._op, core.ReindexOp) and g.shape == x.shape and g._op.overflow_value == 0
    g = jt.grad(x.sum([1, 3]).sum(), x)                    # reduce -> broadcast (of the ones seed)
    assert g.shape == x.shape and isinstance(g._op, core.BroadcastOp)
    s = jt.array(np.zeros((3, 1, 1), np.float32))
    g = jt.grad((x * s).sum(), s)                          # broadcast -> reduce add
    assert g.shape == [3, 1, 1] and isinstance(g._op, core.ReduceOp) and g._op.op == "add"
    # only float targets and losses; untouched targets get zeros of their shape
    with pytest.raises(ValueError):
        jt.grad(x.sum(), jt.array([1, 2]))
    z = jt.grad(x.sum(), s)
    assert z.shape == s.shape
    # history is dropped by stop_grad and under no_grad
    assert (x * 2).stop_grad()._history is None
    with jt.no_grad():
        assert (x * 2)._history is None
    # the gradient of a reshape is the reshape back (ops/reshape_op.cc): again a reindex that shares memory, no scatter
    g = jt.grad((x.reshape([6, 64]) * 3.0).sum(), x)
    assert isinstance(g._op, core.ReindexOp) and getattr(g._op, "same_memory", False) and g.shape == x.shape


def test_assign_of_a_python_number_leaves_the_shared_scalar_alone():
    """Python numbers are kept as one host Var per value; x.assign(2.0) must rebind x to an array of its own and
    leave that shared Var a plain constant: a later `w * 2.0` does not depend on x (its gradient w.r.t. x is the
    zeros of an untouched target), and the constant stays a by-value scalar without a producing op."""
    import jittor_amd as jt
    from jittor_amd import core
    x = jt.array(np.ones(3, np.float32))
    w = jt.array(np.ones(3, np.float32))
    shared = core._as_var(2.0)
    x.assign(2.0)
    assert core._as_var(2.0) is shared and shared._op is None and shared._history is None
    assert x.shape == [1] and not any(v is x for v in (shared._op.inputs if shared._op else ()))
    loss = (w * 2.0).sum()
    g = jt.grad(loss, [x])[0]
    assert g.shape == x.shape and not isinstance(g._op, (core.ReindexReduceOp, core.ReindexOp))   # zeros, not a gradient path
    z = jt.array(np.zeros(2, np.float32))
    z.assign(2.0)
    assert z._op is None or z._op.inputs == []          # an array of its own, not an alias of x


def test_fused_reduce_descriptor_checks_and_specialisation(compile_only):
    """mjt_fused_reduce: one output var (the reduce input); inputs are full-shape or broadcast along exactly
    the reduced axes (one value per output); the kernel with the prologue compiles for gfx950."""
    L = compile_only
    lib = L.load()
    V, F = L.FusedVar, L.FusedOp

    def desc(mask=0, outputs=1):
        spec = [(0, "float32", 0x1000, 0), (0, "float32", 0x2000, mask), (3, "float32", None, 0), (1, "float32", None, 0),
                (2, "float32", None, 0)]
        if outputs == 2:
            spec[3] = (2, "float32", None, 0)
        va = (V * len(spec))()
        for i, (role, dt_, ptr, m) in enumerate(spec):
            va[i].role, va[i].dtype, va[i].ptr, va[i].bcast_mask = role, L.DTYPE_CODE[dt_], ptr, m
        va[2].fvalue = 0.5
        ops = [(1, "multiply", [0, 1], 3), (1, "add", [3, 2], 4)]
        oa = (F * len(ops))()
        for i, (kind, op, ins, out) in enumerate(ops):
            oa[i].kind, oa[i].op, oa[i].out = kind, L.OP_CODE[op], out
            for j, u in enumerate(ins):
                oa[i].inp[j] = u
        d = L.FusedDesc()
        d.ndim = 2
        d.shape[0], d.shape[1] = 64, 256
        d.n_vars, d.vars, d.n_ops, d.ops = len(spec), va, len(ops), oa
        return d, (va, oa)

    ty = L.tensor(0x3000, "float32", [64])
    d, keep = desc()
    assert lib.mjt_fused_reduce(ctypes.byref(d), ctypes.byref(ty), L.OP_CODE["add"], 0b10) == 0
    assert "_pro" in L.last_kernel() and L.last_kernel().startswith("mjt_reduce_row_add")
    ty0 = L.tensor(0x3000, "float32", [256])
    assert lib.mjt_fused_reduce(ctypes.byref(d), ctypes.byref(ty0), L.OP_CODE["maximum"], 0b01) == 0
    # (the column kernel; when it splits the rows among workgroups, its partial results are folded by the row kernel)
    assert L.last_kernel().startswith("mjt_reduce_col_maximum") or L.last_kernel().startswith("mjt_reduce_row_maximum") and L.last_kernel().endswith("_fold")
    d, keep = desc(mask=0b01)                                    # broadcast along a kept axis
    assert lib.mjt_fused_reduce(ctypes.byref(d), ctypes.byref(ty), L.OP_CODE["add"], 0b10) == -2
    d, keep = desc(mask=0b10)                                    # one value per output: row and column kernels
    assert lib.mjt_fused_reduce(ctypes.byref(d), ctypes.byref(ty), L.OP_CODE["add"], 0b10) == 0
    assert L.last_kernel().startswith("mjt_reduce_row_add") and "_pro" in L.last_kernel()
    d, keep = desc(mask=0b01)
    assert lib.mjt_fused_reduce(ctypes.byref(d), ctypes.byref(ty0), L.OP_CODE["add"], 0b01) == 0
    assert L.last_kernel().startswith("mjt_reduce_col_add") or L.last_kernel().endswith("_fold")
    d, keep = desc(outputs=2)
    assert lib.mjt_fused_reduce(ctypes.byref(d), ctypes.byref(ty), L.OP_CODE["add"], 0b10) == -1
    d, keep = desc()
    assert lib.mjt_fused_reduce(ctypes.byref(d), ctypes.byref(ty0), L.OP_CODE["add"], 0b10) == -1    # y has the wrong size
    assert lib.mjt_fused_reduce(ctypes.byref(d), ctypes.byref(ty), L.OP_CODE["subtract"], 0b10) == -1


def test_callers_build_path_graphs():
    """gather / pad / pool / slicing are one reindex (plus a reduce for pool) with the reference's index
    strings (misc.py:1617-1640, nn.py:1679-1700, pool.py:200-208)."""
    import jittor_amd as jt
    from jittor_amd import core
    x = jt.array(np.zeros((2, 3, 8, 8), np.float32))
    g = x.gather(1, jt.array(np.zeros((2, 3, 8, 8), np.int32)))
    assert isinstance(g._op, core.ReindexOp) and g._op.indexes == ["i0", "@e0(i0,i1,i2,i3)", "i2", "i3"]
    p = jt.pad(x, (1, 2), "reflect")
    assert p.shape == [2, 3, 8, 11] and p._op.indexes[3] == "i3<1 ? 1-i3 : i3 > 8 ? 15-i3 : i3-1"
    y = jt.pool(x, 3, "maximum", 1, 2)
    assert isinstance(y._op, core.ReduceOp) and y.shape == [2, 3, 4, 4]
    assert y._history[1][0]._op.indexes == ["i0", "i1", "i2*2-1+i4", "i3*2-1+i5"]
    s = x[1, :, ::2, 3]
    assert s.shape == [3, 4] and s._op.indexes == ["1", "0+i0*(1)", "0+i1*(2)", "3"]
    with pytest.raises(ValueError):
        x.reshape(5, -1)
    with pytest.raises(ValueError):
        jt.pad(x, (1, 2), "mirror")


def test_executor_partitions_a_normalisation_into_three_kernels(monkeypatch):
    """mean, variance (reduce with the subtraction and the square as prologue) and one element-wise kernel:
    `+ eps` and `sqrt` act on the small variance and are evaluated behind their broadcast, and the
    subtraction waits for the division's stage (python/jittor/test/test_new_fused_op.py:24-40 counts the same
    three kernels).  The launches are replaced by recorders: no device is needed."""
    import jittor_amd as jt
    from jittor_amd import executor
    log = []

    def run_group(members, consumers, target_ids, reduce=None, pre=None):
        ids = {m.id for m in members}
        log.append(("group", [getattr(m, "op", m.kind) for m in members], reduce is not None,
                    sorted(getattr(q, "op", q.kind) for m in members for q in (pre or {}).get(m.id, ()))))
        if reduce is not None:
            reduce.out._buf = object()
        for m in members:
            if m.out.id in target_ids or any(c.id not in ids for c in consumers.get(m.out.id, ())):
                m.out._buf = object()
        return True

    def run_single(op):
        log.append(("single", getattr(op, "op", op.kind)))
        op.out._buf = object()

    monkeypatch.setattr(executor, "_run_group", run_group)
    monkeypatch.setattr(executor, "_run_single", run_single)
    v = jt.array(np.zeros((33, 7, 130), np.float32))
    v._buf = object()
    mean = v.mean([2], keepdims=True)
    var = ((v - mean) * (v - mean)).mean([2], keepdims=True)
    y = (v - mean) / (var + 1e-5).sqrt()
    executor._execute(executor._pending_ops([y]), {y.id})
    assert log[0] == ("single", "mean")
    assert log[1][0] == "group" and log[1][2] and log[1][1].count("subtract") == 2 and "multiply" in log[1][1]
    assert log[2][0] == "group" and not log[2][2] and log[2][1][-1] == "divide" and "subtract" in log[2][1]
    assert log[2][3] == ["add", "broadcast", "sqrt"] and len(log) == 3
    # both rules can be switched off
    log.clear()
    monkeypatch.setitem(executor.flags, "enable_broadcast_sink", False)
    v2 = jt.array(np.zeros((4, 6), np.float32))
    v2._buf = object()
    s = v2.sum([1], keepdims=True)
    z = v2 / (s + 1.0)
    executor._execute(executor._pending_ops([z]), {z.id})
    assert [e[0] for e in log] == ["single", "group", "group"]      # sum, s + 1, division


def test_matmul_entry_checks(compile_only):
    """mjt_matmul validates like the reference's relay op (cublas_matmul_op.cc:34-52): 2-d float operands of one
    dtype, matching inner extents, result [n, k]."""
    L = compile_only
    lib = L.load()
    t = lambda dt, shape: L.tensor(0x1000, dt, shape)
    call = lambda a, b, c, ta=0, tb=0: lib.mjt_matmul(ctypes.byref(a), ctypes.byref(b), ctypes.byref(c), ta, tb)
    assert call(t("float32", [4, 8]), t("float32", [8, 5]), t("float32", [4, 5])) == 0
    assert call(t("float32", [8, 4]), t("float32", [8, 5]), t("float32", [4, 5]), 1, 0) == 0
    assert call(t("float32", [4, 8]), t("float32", [5, 8]), t("float32", [4, 5]), 0, 1) == 0
    assert call(t("bfloat16", [4, 8]), t("bfloat16", [8, 5]), t("float32", [4, 5])) == 0
    assert call(t("float32", [4, 8]), t("float32", [7, 5]), t("float32", [4, 5])) == -1
    assert call(t("float32", [4, 8]), t("float32", [8, 5]), t("float32", [5, 4])) == -1
    assert call(t("float32", [4, 8]), t("float16", [8, 5]), t("float32", [4, 5])) == -1
    assert call(t("int32", [4, 8]), t("int32", [8, 5]), t("int32", [4, 5])) == -1
    assert call(t("float32", [4, 8, 1]), t("float32", [8, 5]), t("float32", [4, 5])) == -1
    assert call(t("float32", [3, 4, 8]), t("float32", [3, 8, 5]), t("float32", [3, 4, 5])) == 0       # equal batch extents
    assert call(t("float32", [3, 4, 8]), t("float32", [2, 8, 5]), t("float32", [3, 4, 5])) == -1
    assert lib.mjt_matmul_available() in (0, 1)


def test_shutdown_forgets_kernels_and_rebinding_compiles_again(compile_only, monkeypatch):
    """mjt_shutdown unloads every kernel module; the per-op look-up tables must not keep pointers to them: the same
    calls after binding again have to find (compile or load) their kernels anew."""
    lib = L.load()
    P = 0x100000
    monkeypatch.setenv("MJT_NO_DISK_CACHE", "1")            # count real compilations
    lib.mjt_shutdown()                                       # start from empty tables whatever ran before
    L._device = None
    L.init(-1)

    def calls():
        x, y = L.tensor(P, "float32", (64, 128)), L.tensor(P, "float32", (64,))
        assert lib.mjt_reduce(ctypes.byref(x), ctypes.byref(y), L.OP_CODE["add"], 2) == 0
        xb, w = L.tensor(P, "bfloat16", (2, 64, 16, 16)), L.tensor(P, "bfloat16", (64, 64, 3, 3))
        yb, p = L.tensor(P, "float32", (2, 64, 16, 16)), L.ConvParams(1, 1, 1, 1, 1, 1)
        assert lib.mjt_conv2d_meta(ctypes.byref(xb), ctypes.byref(w), ctypes.byref(yb), ctypes.byref(p)) == 0
        assert L.last_kernel().startswith("mjt_conv_mfma_bf16")
        z = L.tensor(P, "float32", (128, 64))
        assert lib.mjt_reindex(ctypes.byref(x), ctypes.byref(z), 2, L.c_strings(["i1", "i0"]), 0.0, 0, L.c_strings([]), 0, None) == 0
        return L.jit_stats()

    before = L.jit_stats()[0]
    first = calls()[0]
    assert first >= before + 3                               # reduce, convolution (+ its repack), transpose
    assert calls()[0] == first                               # second time: everything from the look-up tables
    lib.mjt_shutdown()
    L._device = None
    L.init(-1)
    assert calls()[0] >= first + 3                           # compiled again, not taken from a stale table


def test_conv_input_gradient_entry_validates_and_picks_its_path(compile_only, monkeypatch):
    """mjt_conv2d_meta_dgrad without a device: argument checks, and which of its five forms a geometry takes (16 bits at strides 1 and 2 one kernel for
    all stride phases, transposed flipped weights for stride 1, few multiply-adds a result at a time, one convolution per stride phase, dy spread out with
    zeros otherwise), by the name of the kernel that runs."""
    lib = L.load()
    P = 0x100000

    def call(xs, ws, params, dys=None, dtype="bfloat16", out=None):
        N, C, H, W = xs
        K, _, R, S = ws
        sh, sw, ph, pw, dh, dw = params
        oh, ow = (H + 2 * ph - dh * (R - 1) - 1) // sh + 1, (W + 2 * pw - dw * (S - 1) - 1) // sw + 1
        dy, w = L.tensor(P, dtype, dys or (N, K, oh, ow)), L.tensor(P, dtype, ws)
        dx, p = L.tensor(P, out or dtype, xs), L.ConvParams(*params)
        return lib.mjt_conv2d_meta_dgrad(ctypes.byref(dy), ctypes.byref(w), ctypes.byref(dx), ctypes.byref(p))

    assert call((2, 64, 28, 28), (64, 64, 3, 3), (2, 2, 1, 1, 1, 1)) == 0
    assert L.last_kernel().startswith("mjt_conv_mfma_bf16_dgrad_c"), L.last_kernel()
    assert call((2, 64, 28, 28), (64, 64, 3, 3), (1, 1, 1, 1, 1, 1)) == 0
    assert L.last_kernel().startswith("mjt_conv_mfma_bf16") and "_dgrad_c" not in L.last_kernel(), L.last_kernel()
    assert call((2, 64, 27, 28), (64, 64, 3, 3), (2, 2, 1, 1, 1, 1)) == 0          # 27 rows: phases of unequal height
    assert L.last_kernel().startswith("mjt_conv_mfma_bf16_dgrad_c"), L.last_kernel()
    for rows, dtype, params in ((28, "float32", (2, 2, 1, 1, 1, 1)), (27, "bfloat16", (3, 3, 0, 0, 1, 1))):
        assert call((2, 64, rows, rows), (64, 64, 3, 3), params, dtype=dtype) == 0
        assert L.last_kernel().startswith("conv_dgrad_phases:"), L.last_kernel()
        assert call((2, 64, rows + 1, rows), (64, 64, 3, 3), params, dtype=dtype) == 0     # no whole phases
        assert not L.last_kernel().startswith("conv_dgrad_phases:") and "_dgrad_c" not in L.last_kernel(), L.last_kernel()
    for rows in (10, 11):                                      # few multiply-adds, with and without whole phases
        assert call((2, 8, rows, 12), (6, 8, 3, 3), (2, 2, 1, 1, 1, 1), dtype="float32") == 0
        assert L.last_kernel().startswith("mjt_conv_direct_dgrad_float32"), L.last_kernel()
        with monkeypatch.context() as m:
            m.setenv("MJT_CONV_DGRAD_NO_DIRECT", "1")
            assert call((2, 8, rows, 12), (6, 8, 3, 3), (2, 2, 1, 1, 1, 1), dtype="float32") == 0
            assert L.last_kernel().startswith("conv_dgrad_phases:" if rows == 10 else "mjt_conv_direct_float32"), L.last_kernel()
    assert call((2, 64, 28, 28), (64, 64, 3, 3), (2, 2, 1, 1, 1, 1), dys=(2, 64, 15, 14)) == -1
    assert b"dy shape" in lib.mjt_last_error()
    assert call((2, 64, 28, 28), (64, 32, 3, 3), (2, 2, 1, 1, 1, 1)) == -1         # weight channels != dx channels
    assert call((2, 64, 28, 28), (64, 64, 1, 1), (1, 1, 1, 1, 1, 1)) == -1         # padding no tap reaches
    assert b"padding" in lib.mjt_last_error()
    assert call((2, 8, 12, 12), (6, 8, 1, 1), (3, 3, 0, 0, 1, 1), out="float32") == 0      # phases that no tap reaches, in the result's type
    for rows, cols, dys in ((0, 9, (2, 6, 1, 6)), (4, 0, (2, 6, 3, 1))):         # a dx of no elements whose dy has some: refused, nothing is launched
        assert call((2, 8, rows, cols), (6, 8, 3, 3), (2, 2, 2, 2, 1, 1), dys=dys, dtype="float32") == -1
        assert b"empty output" in lib.mjt_last_error()


def test_conv_builds_that_ran_out_of_registers_are_not_run(compile_only):
    """The MFMA convolution keeps loads under way in registers the compiler does not track, which is sound only while the
    compiler moves no register aside.  The library reads each build's register figures from the code object: a geometry
    whose build stays within a wave's registers runs on the kernel (among them 32 output channels on two waves and 4-column
    maps, whose builds once did not), one whose build needs more takes another route (the weight-gradient kernel on rows of
    104 columns).  That the first group names the MFMA kernel also shows that the figures are found at all: a build whose
    figures are missing is not run either."""
    lib = L.load()
    P = 0x100000

    def call(xs, ws, params=(1, 1, 1, 1, 1, 1)):
        N, C, H, W = xs
        K, _, R, S = ws
        sh, sw, ph, pw, dh, dw = params
        oh, ow = (H + 2 * ph - dh * (R - 1) - 1) // sh + 1, (W + 2 * pw - dw * (S - 1) - 1) // sw + 1
        x, w, y = L.tensor(P, "bfloat16", xs), L.tensor(P, "bfloat16", ws), L.tensor(P, "bfloat16", (N, K, oh, ow))
        p = L.ConvParams(*params)
        assert lib.mjt_conv2d_meta(ctypes.byref(x), ctypes.byref(w), ctypes.byref(y), ctypes.byref(p)) == 0
        return L.last_kernel()

    assert call((2, 64, 16, 16), (32, 64, 3, 3)).startswith("mjt_conv_mfma_bf16")
    assert call((2, 64, 16, 16), (64, 64, 3, 3)).startswith("mjt_conv_mfma_bf16")
    assert call((2, 32, 40, 4), (64, 32, 3, 3)).startswith("mjt_conv_mfma_bf16")
    # the weight gradient kernel likewise: rows of 104 columns need more registers than there are
    x, dy = L.tensor(P, "bfloat16", (4, 64, 10, 104)), L.tensor(P, "bfloat16", (4, 64, 10, 104))
    dw, p = L.tensor(P, "float32", (64, 64, 3, 3)), L.ConvParams(1, 1, 1, 1, 1, 1)
    assert lib.mjt_conv2d_meta_wgrad(ctypes.byref(x), ctypes.byref(dy), ctypes.byref(dw), ctypes.byref(p)) == -2
    assert b"registers" in lib.mjt_last_error()
    x, dy = L.tensor(P, "bfloat16", (4, 64, 16, 16)), L.tensor(P, "bfloat16", (4, 64, 16, 16))
    assert lib.mjt_conv2d_meta_wgrad(ctypes.byref(x), ctypes.byref(dy), ctypes.byref(dw), ctypes.byref(p)) == 0
    assert L.last_kernel().startswith("mjt_conv_wgrad_mfma_bf16")


def test_plans_of_strided_convolutions_are_not_worked_out_anew(compile_only):
    """Host time of a call on large maps: no walk over their tiles after the first, whether the kernel of windows takes the call or not.  (It was
    19 to 50 times that of a small map; the bound leaves room for a busy machine.)"""
    L, lib = compile_only, compile_only.load()

    def least(call, n, c, size, k, r):
        o = (size - 1) // 2 + 1
        x, w, y = L.tensor(P, "bfloat16", [n, c, size, size]), L.tensor(P, "bfloat16", [k, c, r, r]), L.tensor(P, "bfloat16", [n, k, o, o])
        p = L.ConvParams(2, 2, r // 2, r // 2, 1, 1)
        a = [ctypes.byref(q) for q in ((x, w, y, p) if call == "mjt_conv2d_meta" else (y, w, x, p))]
        times = []
        for _ in range(30):
            t = time.perf_counter()
            L.check(getattr(lib, call)(*a))
            times.append(time.perf_counter() - t)
        return min(times), L.last_kernel()
    small, kern = least("mjt_conv2d_meta", 4, 64, 28, 64, 3)
    assert "_strided_" in kern
    for shape, strided in (((64, 32, 224, 64, 3), False), ((64, 64, 112, 64, 3), False), ((64, 256, 112, 512, 1), True)):
        took, kern = least("mjt_conv2d_meta", *shape)
        assert ("_strided_" in kern) == strided and took < 6 * small + 10e-6, (shape, kern, took, small)
    small, kern = least("mjt_conv2d_meta_dgrad", 4, 64, 28, 64, 3)
    assert "_dgrad_" in kern
    took, kern = least("mjt_conv2d_meta_dgrad", 64, 32, 224, 64, 3)
    assert "_dgrad_" in kern and took < 6 * small + 10e-6, (took, small)


def test_scatter_and_gather_entries_pick_their_kernels(compile_only, monkeypatch):
    """Without a device: which kernel skeleton a reindex_reduce, a reindex and a fused gather + reduce take.  A scatter
    through a window pattern is a gather over x unless it has overflow conditions, extras or too many candidate windows
    per element; a gather into rows that are no whole vectors keeps 16-byte stores; axis permutations go through tiles."""
    lib = L.load()
    P = 0x100000
    e, noex = L.c_strings([]), (L.Tensor * 1)()

    def scatter(ys, xs, idx, op="add", ofc=(), dtype="float32"):
        ty, tx = L.tensor(P, dtype, ys), L.tensor(P, dtype, xs)
        rc = lib.mjt_reindex_reduce(ctypes.byref(ty), ctypes.byref(tx), L.OP_CODE[op], len(idx), L.c_strings(idx), len(ofc),
                                    L.c_strings(list(ofc)), 0, noex)
        assert rc == 0, lib.mjt_last_error()
        return L.last_kernel()

    pool = ([4, 8, 16, 16, 3, 3], [4, 8, 32, 32], ["i0", "i1", "i2*2+i4-1", "i3*2+i5-1"])
    assert scatter(*pool).startswith("mjt_window_scatter_add_")
    assert scatter(*pool, op="maximum", dtype="bfloat16").startswith("mjt_window_scatter_maximum_")
    assert scatter(*pool, ofc=["i4>1"]).startswith("mjt_reindex_reduce_add_")                      # an overflow condition
    assert scatter(*pool, op="bitwise_or", dtype="int32").startswith("mjt_reindex_reduce_bitwise_or_")
    assert scatter([4, 8, 30, 30, 7, 7], [4, 8, 36, 36], ["i0", "i1", "i2+i4", "i3+i5"]).startswith("mjt_reindex_reduce_add_")   # 49 windows reach an element
    assert scatter([4, 8, 16, 16, 3, 3], [4, 8, 32, 32], ["i0", "i1", "i3*2+i4-1", "i2*2+i5-1"]).startswith("mjt_reindex_reduce_add_")  # rows from the column axis
    monkeypatch.setenv("MJT_NO_WINDOW_SCATTER", "1")
    assert scatter(*pool).startswith("mjt_reindex_reduce_add_")
    monkeypatch.delenv("MJT_NO_WINDOW_SCATTER")

    def gather(xs, ys, idx):
        tx, ty = L.tensor(P, "float32", xs), L.tensor(P, "float32", ys)
        assert lib.mjt_reindex(ctypes.byref(tx), ctypes.byref(ty), len(idx), L.c_strings(idx), 0.0, 0, e, 0, noex) == 0, lib.mjt_last_error()
        return L.last_kernel()

    assert gather([8, 16, 64, 64], [8, 64, 64, 16], ["i0", "i3", "i1", "i2"]).startswith("mjt_permute_b4_")
    flat = gather([8, 16, 64, 64], [8, 16, 66, 66], ["i0", "i1", "i2-1", "i3-1"])
    monkeypatch.setenv("MJT_REINDEX_NO_FLAT", "1")
    rows = gather([8, 16, 64, 64], [8, 16, 66, 66], ["i0", "i1", "i2-1", "i3-1"])
    monkeypatch.delenv("MJT_REINDEX_NO_FLAT")
    assert flat.startswith("mjt_reindex_") and rows.startswith("mjt_reindex_") and flat != rows      # four elements per lane, or two
    # column matrices with the pixels innermost: per image, the whole batch as one group, chunks of images; a stride the
    # pattern does not have (the image index times 3 for chunks of 2) stays on the generic kernel
    taps = ["i4-1+i2", "i5-1+i3"]
    assert gather([8, 16, 28, 28], [8, 16, 3, 3, 28, 28], ["i0", "i1"] + taps).startswith("mjt_im2col_planes_b4_28x28_k3x3")
    assert gather([8, 16, 7, 7], [16, 3, 3, 8, 7, 7], ["i3", "i0", "i4-1+i1", "i5-1+i2"]).endswith("_n8_v4")
    assert gather([8, 16, 29, 29], [4, 16, 3, 3, 2, 14, 14], ["i0*2+i4", "i1", "i5*2-1+i2", "i6*2-1+i3"]).endswith("_n2_v4")
    assert gather([12, 16, 14, 14], [4, 16, 3, 3, 2, 14, 14], ["i0*3+i4", "i1", "i5-1+i2", "i6-1+i3"]).startswith("mjt_reindex_")

    loop, z = L.tensor(0, "float32", [8, 16, 32, 32, 2, 2]), L.tensor(P, "float32", [8, 16, 32, 32])
    tx = L.tensor(P, "float32", [8, 16, 64, 64])
    assert lib.mjt_reindex_then_reduce(ctypes.byref(tx), ctypes.byref(loop), ctypes.byref(z), L.OP_CODE["maximum"], 2, 4,
                                       L.c_strings(["i0", "i1", "i2*2+i4", "i3*2+i5"]), 0.0, 0, e, 0, noex) == 0
    assert L.last_kernel().startswith("mjt_reindex_then_maximum_")


def test_compile_options_follow_the_flag_and_mark_grouped_convolutions():
    """Var.compile_options (var_holder.h:265-273): a dict name -> int, initialised from the flag's value when the var is
    created (var.cc:75); nn.conv2d marks the gathered input of a grouped convolution with {"G": groups} (nn.py:1278),
    and the mark does not stand in the way of the matcher."""
    import jittor_amd.executor as E
    assert jt.zeros([2]).compile_options == {}
    with jt.flag_scope(compile_options={"parallel": 0}):
        v = jt.zeros([2])
    assert v.compile_options == {"parallel": 0} and jt.zeros([2]).compile_options == {}
    v.compile_options = {"G": 4, "C": 8}
    assert v.compile_options == {"G": 4, "C": 8}
    got = v.compile_options
    got["G"] = 5                                       # a copy: the var keeps its own
    assert v.compile_options["G"] == 4
    with pytest.raises(TypeError):
        v.compile_options = {"G": 1.5}
    x, w = jt.zeros([1, 8, 6, 6]), jt.zeros([8, 2, 3, 3])
    y = jt.nn.conv2d(x, w, padding=1, groups=4)
    scatter = y._op
    product = scatter.inputs[0]._op
    assert product.inputs[0].compile_options == {"G": 4}
    unit = E._match_conv_grouped(scatter)
    assert unit is not None and unit.groups == 4


def test_conv_gradient_patterns_match_for_common_losses():
    """The two backward patterns are recognised whatever stands between the convolution and the loss: the loss may
    be the output itself (jt.grad seeds ones, test_conv_tuner.py:105-133), its sum or mean (for 16-bit outputs these
    put float32 casts around dy: the narrowing cast of dy stays, the identity casts are looked through) or a product."""
    from jittor_amd import executor as E
    for dtype in ("float32", "float16", "bfloat16"):
        x, w = jt.zeros([2, 3, 8, 8]).cast(dtype), jt.zeros([4, 3, 3, 3]).cast(dtype)
        y = jt.nn.conv2d(x, w, padding=1)
        r = jt.zeros(y.shape).cast(dtype)
        for loss in (y, y.sum(), y.mean(), (y * r).sum(), (y * y).sum()):
            gx, gw = jt.grad(loss, [x, w])
            ux, uw = E._match_conv_bwd(gx._op), E._match_conv_bwd(gw._op)
            assert isinstance(ux, E.ConvBwdDataUnit) and isinstance(uw, E.ConvBwdWeightUnit), (dtype, loss)
            assert ux.inputs[0].dtype == dtype and list(ux.inputs[0].shape) == [2, 4, 8, 8]
            assert uw.inputs[1].dtype == dtype and gx.dtype == dtype and gw.dtype == dtype


def test_grouped_conv_and_its_gradients_are_matched_by_role():
    """Over the grouped form's 8-d product each of x, w and y has its own index pattern; the scattered-into one names
    the unit.  Forward, input gradient and weight gradient of a grouped and of a depthwise convolution are recognised,
    with the geometry read back from the x pattern."""
    from jittor_amd import executor as E
    for dtype in ("float32", "bfloat16"):
        for groups, cin, cout, kw in ((2, 4, 6, dict(padding=1)), (4, 4, 4, dict(stride=2, padding=1)), (3, 6, 3, dict(padding=2, dilation=2))):
            x, w = jt.zeros([2, cin, 9, 8]).cast(dtype), jt.zeros([cout, cin // groups, 3, 3]).cast(dtype)
            y = jt.nn.conv2d(x, w, groups=groups, **kw)
            r = jt.zeros(y.shape).cast(dtype)
            fwd = E._match_conv_grouped(y._op)
            assert isinstance(fwd, E.ConvUnit) and fwd.groups == groups and fwd.inputs[0] is x and fwd.inputs[1] is w
            gx, gw = jt.grad((y * r).sum(), [x, w])
            ux, uw = E._match_conv_grouped(gx._op), E._match_conv_grouped(gw._op)
            assert isinstance(ux, E.ConvBwdDataUnit) and isinstance(uw, E.ConvBwdWeightUnit), (dtype, groups)
            assert ux.groups == groups and uw.groups == groups and ux.params == fwd.params and uw.params == fwd.params
            assert ux.inputs[1] is w and uw.inputs[0] is x
            assert list(ux.inputs[0].shape) == list(y.shape) and ux.inputs[0] is uw.inputs[1]
            assert gx.dtype == dtype and gw.dtype == dtype
    # an 8-d scatter-add that is none of the three stays what it is
    a = jt.zeros([2, 2, 3, 2, 4, 4, 3, 3])
    z = (a * a).reindex_reduce("add", [2, 6, 4, 4], ["i0", "i1*3+i2", "i5", "i4"])
    assert E._match_conv_grouped(z._op) is None


def test_executor_replays_a_graph_it_has_seen(compile_only, monkeypatch):
    """The second execution of a graph with the same signature re-issues the recorded library calls: same number of calls
    and the same counters, every pointer inside the recorded descriptors is the new graph's (input, result or a buffer
    made on the way), a by-value scalar is the new graph's value, computed vars become leaves; another shape, another
    wiring or a switched flag is another signature.  Compile-only mode with addresses handed out by a counter: no device."""
    from jittor_amd import core, executor
    nxt = [0x10000000]

    def fake_alloc(nbytes):
        size = core._Pool._round(nbytes)
        nxt[0] += size
        return nxt[0] - size, size

    monkeypatch.setattr(core.pool, "alloc", fake_alloc)
    monkeypatch.setattr(core.pool, "free", lambda ptr, size: None)
    monkeypatch.setattr(L, "h2d", lambda ptr, arr: None)
    monkeypatch.setitem(executor.flags, "enable_replay", True)
    executor._plans.clear()

    def step(lr, shape=(3, 6, 10, 10), twice=False):
        x = jt.array(np.ones(shape, np.float32))
        w = jt.array(np.ones((8, shape[1], 3, 3), np.float32))
        y = jt.nn.conv2d(x, w, padding=1)
        gw, = jt.grad((y * y).sum(), [w])                    # float32 weight gradient: column matrices and partial sums on the way
        new_w = w - gw * jt.array(np.float32(lr))            # a by-value scalar
        flat = jt.reshape(y, [shape[0], -1])                 # shares y's buffer
        out = (flat + flat) if twice else (flat + 1.0)
        before = dict(executor.stats)
        jt.sync([new_w, out, y])
        return {k: executor.stats[k] - before[k] for k in before}, (x, w, y, new_w, out, flat)

    d1, keep1 = step(0.5)
    assert d1["plans"] == 1 and d1["replays"] == 0
    plan = next(iter(executor._plans.values()))
    ncalls = len(plan.calls)
    d2, keep2 = step(0.25)
    assert d2["replays"] == 1 and d2["plans"] == 0
    for k in d1:
        if k not in ("plans", "replays"):
            assert d1[k] == d2[k], k
    assert len(plan.calls) == ncalls and ncalls == d1["launches"]
    # every recorded pointer now points into a buffer of the second graph (or one made during the replay), none into the first's
    x1, w1, y1, nw1, out1, flat1 = keep1
    x2, w2, y2, nw2, out2, flat2 = keep2
    first = {v._buf.ptr for v in keep1}
    second = {v._buf.ptr for v in keep2}
    assert not first & second and flat2._buf is y2._buf and flat1._buf is y1._buf
    seen = set()
    for obj, idx, slot, off in plan.ptrs:
        ptr = (obj if idx is None else obj[idx]).ptr
        assert ptr - off not in first
        seen.add(ptr - off)
    assert second - {flat2._buf.ptr} <= seen | {y2._buf.ptr}
    assert all(v._op is None for v in (y2, nw2, out2))
    vals = [arr[i].fvalue for arr, i, _ in plan.scalars]
    assert 0.25 in vals and 0.5 not in vals
    # other signatures: a shape, the wiring of a leaf, a flag
    assert step(0.5, shape=(3, 6, 12, 10))[0]["plans"] == 1
    assert step(0.5, twice=True)[0]["plans"] == 1
    monkeypatch.setitem(executor.flags, "enable_reduce_fusion", False)
    assert step(0.5)[0]["plans"] == 1
    monkeypatch.setitem(executor.flags, "enable_replay", False)
    d = step(0.5)[0]
    assert d["plans"] == 0 and d["replays"] == 0


def test_recorded_launches(compile_only, monkeypatch):
    """From its third execution on a graph's launches are issued by one call; what cannot be recorded (a scatter that keeps
    tallies) stays with its calls, a recording older than a shutdown is refused and made again, two recordings of different
    work are not matched."""
    from jittor_amd import core, executor
    nxt = [0x10000000]

    def fake_alloc(nbytes):
        size = core._Pool._round(nbytes)
        nxt[0] += size
        return nxt[0] - size, size

    monkeypatch.setattr(core.pool, "alloc", fake_alloc)
    monkeypatch.setattr(core.pool, "free", lambda ptr, size: None)
    monkeypatch.setattr(L, "h2d", lambda ptr, arr: None)
    monkeypatch.setitem(executor.flags, "enable_replay", True)
    executor._plans.clear()

    def norm(scale):
        x = jt.array(np.ones((64, 48), np.float32))
        d = x - x.mean([1], keepdims=True)
        jt.sync([d * jt.array(np.float32(scale)), (d * d).sum([0])])

    def scatter(_):
        v, i = jt.array(np.ones(1 << 20, np.float32)), jt.array(np.zeros(1 << 20, np.int32))
        jt.sync([v.reindex_reduce("add", [1 << 18], ["@e0(i0)"], extras=[i])])

    def recorded(step, n):
        before = executor.stats["recorded_launches"]
        for k in range(n):
            step(1.0 + k)
        return executor.stats["recorded_launches"] - before

    assert recorded(norm, 2) == 0 and recorded(norm, 3) == 3
    plan = next(iter(executor._plans.values()))
    assert plan.native and all((o if i is None else o[i]).ptr is not None for o, i, _, _ in plan.ptrs)
    assert recorded(scatter, 4) == 0
    L.load().mjt_shutdown()
    L.check(L.load().mjt_init(-1))
    assert recorded(norm, 2) == 1                                # refused once, recorded anew
    lib = L.load()
    recs = []
    for shape in ([64, 48], [64, 40]):
        x, y = L.tensor(1 << 45, "float32", shape), L.tensor(1 << 46, "float32", [64])
        L.check(lib.mjt_record_begin())
        assert lib.mjt_record_begin() < 0                        # one at a time
        L.check(lib.mjt_reduce(ctypes.byref(x), ctypes.byref(y), L.OP_CODE["add"], 2))
        rec = ctypes.c_void_p()
        L.check(lib.mjt_record_end(ctypes.byref(rec)))
        recs.append(rec)
    b, b2 = (ctypes.c_uint64 * 2)(1 << 45, 1 << 46), (ctypes.c_uint64 * 2)(1 << 47, 1 << 48)
    none = (ctypes.c_int64 * 1)()
    assert lib.mjt_record_relocate(recs[0], recs[1], 2, b, b, 1 << 36, 0, none, none) not in (0, L.ERR_UNSUPPORTED)   # one address in both
    assert lib.mjt_record_relocate(recs[0], recs[1], 2, b, b2, 1 << 36, 0, none, none) == L.ERR_UNSUPPORTED
    assert lib.mjt_record_launch(recs[0], 2, b, 0, None, none) < 0
    for rec in recs:
        lib.mjt_record_free(rec)


def test_recording_refuses_what_is_no_launch_of_its_own(compile_only):
    """Copies to and from host memory, events and the two calls of where act on the device, or on the host, the moment they are
    made: between begin and end, where addresses may be stand-ins, they are refused.  Nothing to do is nothing to refuse."""
    lib = L.load()
    count, host = ctypes.c_int64(), ctypes.create_string_buffer(64)
    cond, empty, out = L.tensor(1 << 45, "float32", [64]), L.tensor(1 << 45, "float32", [0]), (L.Tensor * 1)(L.tensor(1 << 46, "int32", [64]))
    none = (L.Tensor * 1)(L.tensor(1 << 46, "int32", [0]))
    dev = ctypes.c_void_p(1 << 45)
    L.check(lib.mjt_record_begin())
    try:
        for name, rc in (("where_count", lib.mjt_where_count(ctypes.byref(cond), ctypes.byref(count))),
                         ("where", lib.mjt_where(ctypes.byref(cond), 64, out)),
                         ("h2d", lib.mjt_h2d(dev, host, 64)), ("d2h", lib.mjt_d2h(host, dev, 64)), ("event", lib.mjt_event_record(None))):
            assert rc == L.ERR_UNSUPPORTED and "recording" in lib.mjt_last_error().decode(), name
        assert lib.mjt_where_count(ctypes.byref(empty), ctypes.byref(count)) == 0 and count.value == 0
        assert lib.mjt_where(ctypes.byref(empty), 0, none) == 0
    finally:
        L.check(lib.mjt_record_end(None))
    assert lib.mjt_where_count(ctypes.byref(cond), ctypes.byref(count)) == 0
    assert lib.mjt_where(ctypes.byref(cond), 64, out) == 0


@pytest.mark.parametrize("pairs", [1, 170, 171, 172, 400])
def test_recorded_launches_tell_all_buffers_apart(compile_only, monkeypatch, pairs):
    """The two sets of stand-in addresses share none, also where a graph has more buffers (3 per pair) than fit between two
    powers of two: a buffer with one address in both would be recorded as a constant."""
    from jittor_amd import core, executor
    nxt = [0x10000000]

    def fake_alloc(nbytes):
        size = core._Pool._round(nbytes)
        nxt[0] += size
        return nxt[0] - size, size

    monkeypatch.setattr(core.pool, "alloc", fake_alloc)
    monkeypatch.setattr(core.pool, "free", lambda ptr, size: None)
    monkeypatch.setattr(L, "h2d", lambda ptr, arr: None)
    monkeypatch.setitem(executor.flags, "enable_replay", True)
    executor._plans.clear()
    lib, sets = L.ensure_init(), []

    class Library:
        def __getattr__(self, name):
            return getattr(lib, name)

        def mjt_record_relocate(self, first, second, n, b1, b2, *rest):
            sets.append((list(b1), list(b2)))
            return lib.mjt_record_relocate(first, second, n, b1, b2, *rest)

    monkeypatch.setattr(L, "ensure_init", lambda: Library())
    before = executor.stats["recorded_launches"]
    for _ in range(3):
        keep = [(jt.array(np.ones((4, 4 + k % 2), np.float32)), jt.array(np.ones((4, 4 + k % 2), np.float32))) for k in range(pairs)]
        jt.sync([(a * b).sum([1]) for a, b in keep])
    assert executor.stats["recorded_launches"] == before + 1
    (b1, b2), = sets
    assert len(b1) >= 3 * pairs and len(set(b1 + b2)) == 2 * len(b1)


def test_one_thread_at_a_time_executes_a_plan(compile_only, monkeypatch):
    """A plan's descriptors, which hold stand-in addresses while its launches are recorded, belong to one execution at a time."""
    import threading
    import time
    from jittor_amd import core, executor
    nxt = [0x10000000]

    def fake_alloc(nbytes):
        size = core._Pool._round(nbytes)
        nxt[0] += size
        return nxt[0] - size, size

    monkeypatch.setattr(core.pool, "alloc", fake_alloc)
    monkeypatch.setattr(core.pool, "free", lambda ptr, size: None)
    monkeypatch.setattr(L, "h2d", lambda ptr, arr: None)
    monkeypatch.setitem(executor.flags, "enable_replay", True)
    executor._plans.clear()
    inside, met, failed = [], [], []
    for name in ("_launch", "_record"):
        def watched(*args, _f=getattr(executor, name)):
            me = threading.get_ident()
            met.extend(t for t in inside if t != me)
            inside.append(me)
            time.sleep(0.001)                                          # lets the others run
            try:
                return _f(*args)
            finally:
                inside.remove(me)
        monkeypatch.setattr(executor, name, watched)

    def work():
        try:
            for _ in range(5):
                x = jt.array(np.ones((32, 24), np.float32))
                jt.sync([(x * x).sum([1])])
        except Exception as e:                                         # shown by the assertion below
            failed.append(e)

    work()                                                             # the plan is there
    threads = [threading.Thread(target=work) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed and not met


def _graph_of(v):
    """What v is computed from: its ops in the order of their results, with their inputs by number; leaves by their shape."""
    seen, stack = {}, [v]
    while stack:
        u = stack.pop()
        if u.id not in seen:
            seen[u.id] = u
            stack.extend(u._history[1] if u._history is not None else ())
    order = [seen[k] for k in sorted(seen)]
    number = {u.id: i for i, u in enumerate(order)}
    return [(u._history[0].sig(),) + tuple(number[w.id] for w in u._history[1]) if u._history is not None else tuple(u.shape) for u in order], seen


@pytest.mark.parametrize("scale", [
    lambda x, s: (x * x).sum() * s,                                    # the factor is a leaf of one element
    lambda x, s: ((x * x) * s).sum(),                                  # ... spread inside the graph
    lambda x, s: ((x * x) * s.cast("float64").cast("float32")).sum(),  # ... cast
])
@pytest.mark.parametrize("dtype", ["float32", "float16", "bfloat16"])
def test_second_derivative_by_a_scale_whatever_its_value(scale, dtype):
    """A gradient leaves out the products with its own seed only: a parameter that holds a 1 stays in the graph like any other."""
    graphs = []
    for value in (1.0, 1.5):
        x = jt.array(np.arange(1, 5, dtype=np.float32), dtype)
        s = jt.array(np.array([value], np.float32), dtype)
        dx = jt.grad(scale(x, s), x)
        graph, seen = _graph_of(dx)
        assert s.id in seen
        ds, seen = _graph_of(jt.grad(dx.sum(), s))
        assert x.id in seen
        graphs.append((graph, ds))
    assert graphs[0] == graphs[1]


def test_products_with_the_seed_are_left_out_unless_the_caller_holds_it():
    x, w = jt.array(np.ones((3, 4), np.float32)), jt.array(np.ones((3, 4), np.float32))
    y = x * w
    gx = jt.grad(y.sum(), x)
    assert gx.id != w.id and _graph_of(gx)[0] == [(3, 4), (("unary", "cast"), 0)]           # w, as a Var of its own
    gx, gy = jt.grad(y.sum(), [x, y])                                    # gy is the seed, spread
    assert gy.id in _graph_of(gx)[1]
    assert w.id in _graph_of(jt.grad(gx.sum(), gy))[1]
    one = jt.grad(x.sum(), x)                                            # a seed of an earlier call is a Var like any other
    a = jt.array(np.ones((3, 4), np.float32))
    da = jt.grad(((a * x) * one).sum(), a)
    assert one.id in _graph_of(da)[1]


class _FakeDriver:
    """Allocations that are only counted; a call lets other threads run, as the driver does."""

    def __init__(self, monkeypatch):
        self.live, self.made, self.on_free = {}, 0, None
        monkeypatch.setattr(L, "alloc", self.alloc)
        monkeypatch.setattr(L, "free", self.free)
        monkeypatch.setattr(L, "device", lambda: 0)

    def alloc(self, size):
        import time
        time.sleep(0)
        self.made += 1
        ptr = object()
        self.live[id(ptr)] = (ptr, size)
        return ptr

    def free(self, ptr):
        import time
        time.sleep(0)
        del self.live[id(ptr)]


@pytest.mark.parametrize("limit", [1 << 40, 5000])
def test_pool_keeps_count_of_its_blocks_between_threads(monkeypatch, limit):
    """Threads that take and give back blocks of a few sizes, with a pool that has room and with one that is always full: no
    error, every block is in the pool or with the driver, and the pool's count is that of its lists."""
    import sys
    import threading
    from jittor_amd import core
    driver, pool, failed = _FakeDriver(monkeypatch), core._Pool(), []
    pool.limit = limit
    every = sys.getswitchinterval()
    sys.setswitchinterval(1e-6)

    def work(seed):
        rng = np.random.default_rng(seed)
        held = []
        try:
            for size in rng.choice([256, 512, 1024, 4096], 8000):
                held.append(pool.alloc(int(size)))
                if len(held) > 3:
                    pool.free(*held.pop(0))
            for block in held:
                pool.free(*block)
        except Exception as e:                                         # shown by the assertion below
            failed.append(repr(e))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    try:
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    finally:
        sys.setswitchinterval(every)
    assert not failed, failed[:3]
    cached = [(id(p), size) for size, lst in pool.free_blocks.items() for p in lst]
    assert len(set(cached)) == len(cached) and sorted(cached) == sorted((k, size) for k, (_, size) in driver.live.items())
    assert pool.cached_bytes == sum(size for _, size in cached) <= limit
    assert all(pool.free_blocks.values())
    pool.release_all()
    assert not driver.live and pool.cached_bytes == 0


@pytest.mark.parametrize("first,second", [(256, 256), (256, 512), (512, 256)])
def test_pool_takes_blocks_back_from_a_finaliser_inside_its_own_bookkeeping(monkeypatch, first, second):
    """A collection may start while a block is taken in and drop another one: both are kept, and counted."""
    from jittor_amd import core
    driver, pool = _FakeDriver(monkeypatch), core._Pool()
    blocks, late = [pool.alloc(first), pool.alloc(first)], [pool.alloc(second)]

    class Collecting(dict):
        def pop(self, *args):
            got = dict.pop(self, *args)
            if late and not armed:
                pool.free(*late.pop())                                 # between two steps of the call under way
            return got

    armed = [1]
    pool.free(*blocks[0])
    pool.free_blocks = Collecting(pool.free_blocks)
    armed.clear()
    pool.free(*blocks[1])
    sizes = sorted(size for size, lst in pool.free_blocks.items() for _ in lst)
    assert sizes == sorted([first, first, second]) and pool.cached_bytes == sum(sizes) and len(driver.live) == 3


def test_routes_that_want_workspace_have_one_without(compile_only, monkeypatch):
    """Padded copies of unaligned rows, slices of long sums and slices of a weight gradient are for speed: without the memory for
    them (here: a limit on it) the call runs as it lies, or is handed back to the caller who has another way."""
    lib = compile_only.load()
    p = L.ConvParams(1, 1, 1, 1, 1, 1)

    def product(m, k, n, dt, ta, tb):
        a, b = (L.tensor(P, dt, s) for s in ([k, m] if ta else [m, k], [n, k] if tb else [k, n]))
        c = L.tensor(P, dt, [m, n])
        L.check(lib.mjt_matmul(ctypes.byref(a), ctypes.byref(b), ctypes.byref(c), ta, tb))
        return L.last_kernel()

    def wgrad(dt):
        x, dy, dw = L.tensor(P, dt, [64, 40, 15, 13]), L.tensor(P, dt, [64, 72, 15, 13]), L.tensor(P, "float32", [72, 40, 3, 3])
        rc = lib.mjt_conv2d_meta_wgrad(ctypes.byref(x), ctypes.byref(dy), ctypes.byref(dw), ctypes.byref(p))
        return rc, L.last_kernel()

    monkeypatch.delenv("MJT_MOST_WORKSPACE", raising=False)
    assert product(301, 203, 129, "bfloat16", 0, 0).startswith("mjt_gemm_mfma_")
    assert product(64, 4096, 64, "float32", 1, 0).endswith("_slices")
    for dt in ("float32", "bfloat16"):
        rc, kernel = wgrad(dt)
        assert rc == 0 and kernel.startswith("mjt_conv_wgrad_igemm_")
    monkeypatch.setenv("MJT_MOST_WORKSPACE", "4096")
    for ta in (0, 1):
        for tb in (0, 1):
            assert product(301, 203, 129, "bfloat16", ta, tb).startswith("mjt_gemm_plain_")
    assert product(301, 208, 129, "bfloat16", 0, 0).startswith("mjt_gemm_plain_")          # one operand of the two
    kernel = product(64, 4096, 64, "float32", 1, 0)
    assert kernel.startswith("mjt_gemm_mfma_") and not kernel.endswith("_slices")
    for dt in ("float32", "bfloat16"):
        assert wgrad(dt)[0] == L.ERR_UNSUPPORTED
    monkeypatch.setenv("MJT_MOST_WORKSPACE", str(1 << 30))
    assert product(301, 203, 129, "bfloat16", 0, 0).startswith("mjt_gemm_mfma_")


@pytest.mark.parametrize("what", ["conv", "dgrad"])
@pytest.mark.parametrize("flat", ["0", "1"])
def test_routes_without_a_group_refuse_before_they_prepare(compile_only, monkeypatch, what, flat):
    """A convolution through column matrices takes no group behind it, and says so before it launches anything: neither the copy of its
    weight rows to whole 16 bytes nor, for an input gradient, the transposed weights."""
    lib = compile_only.load()
    monkeypatch.setenv("MJT_CONV_NO_IGEMM", "1")
    monkeypatch.setenv("MJT_CONV_FLAT", flat)
    dt = "float32" if flat == "0" else "bfloat16"              # (the whole-batch product is one of 16 bits)
    code = L.DTYPE_CODE[dt]
    x, w, y = L.tensor(P, dt, [2, 15, 30, 30]), L.tensor(P, dt, [33, 15, 3, 3]), L.tensor(P, dt, [2, 33, 30, 30])
    out = y if what == "conv" else x
    fv = (L.FusedVar * 2)(L.FusedVar(L.VAR_PRODUCT, code, None), L.FusedVar(L.VAR_OUTPUT, code, P))
    fo = (L.FusedOp * 1)(L.FusedOp(L.FOP_UNARY, L.OP_CODE["negative"], (0, 0, 0), 1))
    d = L.FusedDesc(4, tuple(out.shape[:4]), 2, fv, 1, fo)
    p = L.ConvParams(1, 1, 1, 1, 1, 1)
    probe = L.tensor(P, "float32", [64])
    L.check(lib.mjt_reduce(ctypes.byref(probe), ctypes.byref(L.tensor(P, "float32", [1])), L.OP_CODE["add"], 1))
    last = L.last_kernel()
    if what == "conv":
        rc = lib.mjt_conv2d_meta_then(ctypes.byref(x), ctypes.byref(w), ctypes.byref(y), ctypes.byref(p), 1, ctypes.byref(d))
    else:
        rc = lib.mjt_conv2d_meta_dgrad_then(ctypes.byref(y), ctypes.byref(w), ctypes.byref(x), ctypes.byref(p), ctypes.byref(d))
    assert rc == L.ERR_UNSUPPORTED and L.last_kernel() == last
    L.check(lib.mjt_conv2d_meta(ctypes.byref(x), ctypes.byref(w), ctypes.byref(y), ctypes.byref(p)))
    assert L.last_kernel() == ("conv_as_batch_gemm" if flat == "1" else "conv_as_reindex_gemm")


def test_float32_weight_gradient_of_a_few_tiles_is_cut_into_slices(compile_only, monkeypatch):
    """One to thirty tiles and a sum of ten to a hundred stages: small tiles, and as many slices as there are compute units to run
    them (they need workspace, so that a limit on it hands the call back), not one workgroup for the whole sum."""
    lib = compile_only.load()
    for n, c, h, k, r, s in ((64, 64, 7, 64, 1, 1), (16, 100, 9, 70, 3, 2), (4, 64, 14, 64, 3, 1), (18, 48, 14, 82, 1, 1), (16, 256, 14, 256, 1, 1)):
        pad = r // 2
        o = (h + 2 * pad - r) // s + 1
        x, dy, dw = L.tensor(P, "float32", [n, c, h, h]), L.tensor(P, "float32", [n, k, o, o]), L.tensor(P, "float32", [k, c, r, r])
        p = L.ConvParams(s, s, pad, pad, 1, 1)
        monkeypatch.delenv("MJT_MOST_WORKSPACE", raising=False)
        L.check(lib.mjt_conv2d_meta_wgrad(ctypes.byref(x), ctypes.byref(dy), ctypes.byref(dw), ctypes.byref(p)))
        assert L.last_kernel().startswith("mjt_conv_wgrad_igemm_float32") and L.last_kernel().endswith("_64x64")
        monkeypatch.setenv("MJT_MOST_WORKSPACE", "0")
        assert lib.mjt_conv2d_meta_wgrad(ctypes.byref(x), ctypes.byref(dy), ctypes.byref(dw), ctypes.byref(p)) == L.ERR_UNSUPPORTED


def test_products_of_unaligned_rows_are_copied_where_that_pays(compile_only):
    """Short sums run as they lie, unless there is much of them: copying operands into padded rows costs more than such a sum."""
    lib = compile_only.load()

    def kernel(m, k, n, dt, ta, tb):
        a, b = (L.tensor(P, dt, s) for s in ([k, m] if ta else [m, k], [n, k] if tb else [k, n]))
        c = L.tensor(P, dt, [m, n])
        L.check(lib.mjt_matmul(ctypes.byref(a), ctypes.byref(b), ctypes.byref(c), ta, tb))
        return "plain" if L.last_kernel().startswith("mjt_gemm_plain_") else "copied" if L.last_kernel().startswith("mjt_gemm_mfma_") else L.last_kernel()

    for dt in ("float32", "bfloat16", "float16"):
        assert [kernel(m, k, n, dt, 0, 0) for m, k, n in (
            (4097, 17, 65), (1025, 33, 1025), (1025, 47, 257), (20001, 15, 513)           # short sums; below 16 however many
        )] == ["plain"] * 4
        assert [kernel(m, k, n, dt, 0, 0) for m, k, n in (
            (1025, 49, 1025), (4097, 33, 513), (4097, 17, 1025), (101, 97, 129), (129, 4097, 65)
        )] == ["copied"] * 5
        assert kernel(1001, 41, 504, dt, 0, 0) == "copied" and kernel(1001, 41, 505, dt, 0, 0) == "plain"      # one operand copied, both


def test_batches_of_small_unaligned_products_run_as_they_lie(compile_only):
    """Many rows that share little work: copying them into padded rows costs more than the matrix cores save."""
    lib = compile_only.load()

    def copied(batch, m, k, n, dt):
        a, b, c = (L.tensor(P, dt, s) for s in ([batch, m, k], [batch, n, k], [batch, m, n]))
        L.check(lib.mjt_matmul(ctypes.byref(a), ctypes.byref(b), ctypes.byref(c), 0, 1))
        return not L.last_kernel().startswith("mjt_gemm_plain_")

    for dt in ("float32", "bfloat16", "float16"):
        for shape in ((256, 50, 63, 50), (256, 50, 97, 50), (17, 816, 63, 48), (64, 100, 49, 100)):
            assert not copied(*shape, dt), (shape, dt)
        for shape in ((17, 816, 201, 48), (64, 100, 131, 100), (8, 512, 71, 512), (1, 816, 63, 816)):
            assert copied(*shape, dt), (shape, dt)


@pytest.mark.parametrize("k,s,p,dtype", [(2, 2, 0, "bfloat16"), (3, 2, 1, "bfloat16"), (3, 1, 1, "float32"), (4, 1, 0, "float32"),
                                         (2, 1, 0, "float16"), (4, 2, 1, "bfloat16"), (5, 2, 2, "float32")])
def test_window_gradients_bound_what_a_lane_unrolls(compile_only, monkeypatch, k, s, p, dtype):
    """The windows that reach any of a lane's elements, for each of them: the kernel does not compile with more than 40 bodies."""
    from jittor_amd import core, executor
    nxt = [0x10000000]

    def fake_alloc(nbytes):
        size = core._Pool._round(nbytes)
        nxt[0] += size
        return nxt[0] - size, size

    monkeypatch.setattr(core.pool, "alloc", fake_alloc)
    monkeypatch.setattr(core.pool, "free", lambda ptr, size: None)
    monkeypatch.setattr(L, "h2d", lambda ptr, arr: None)
    x = jt.array(np.ones((2, 3, 32, 32), np.float32), dtype)
    y = jt.pool(x, k, "maximum", p, s)
    g = jt.array(np.ones(y.shape, np.float32), dtype)
    jt.sync([x, y, g])
    before = executor.stats["fused_scatters"]
    jt.sync([jt.grad((jt.pool(x, k, "maximum", p, s) * g).sum(), x)])
    assert executor.stats["fused_scatters"] == before + 1


def test_assign_keeps_what_a_program_hung_on_the_var():
    """assign() rebinds the value; attributes that are the program's own stay, and nothing of the old value lingers."""
    w = jt.array(np.float32(3.0)).stop_fuse().name("w")
    w.decay = 0.1
    assert w.is_scalar
    w.assign(jt.array(np.ones((2, 3), np.float32)))
    assert w.decay == 0.1 and w.name() == "w" and w.shape == [2, 3] and not w.is_scalar and not w._stop_fuse
    w.assign(w * 2.0)
    assert w.decay == 0.1 and w.name() == "w" and w._host is None
    w.assign(1.5)
    assert w.decay == 0.1 and w.is_scalar and w.item() == 1.5


def test_dtype_rules_kept_are_those_of_one_register(monkeypatch):
    """Another thread may set the register (a gradient does, op by op) while a rule is worked out: what is kept for a register is
    what that register gives."""
    from jittor_amd import dtypes as dt
    monkeypatch.setattr(dt, "amp_reg", 0)
    monkeypatch.setattr(dt, "_binary_dtypes", {})
    size = dt.dsize_

    def meanwhile(name):
        dt.amp_reg = dt.AMP_PREFER16
        return size(name)

    monkeypatch.setattr(dt, "dsize_", meanwhile)
    assert dt.binary_dtype_infer("add", "float32", "float32") == "float32"
    monkeypatch.setattr(dt, "dsize_", size)
    dt.amp_reg = 0
    assert dt.binary_dtype_infer("add", "float32", "float32") == "float32"
    dt.amp_reg = dt.AMP_PREFER16
    assert dt.binary_dtype_infer("add", "float32", "float32") == "float16"


@pytest.fixture
def fake_buffers(compile_only, monkeypatch):
    """The front end on made-up device addresses, nothing launched; no plans from before."""
    from jittor_amd import core, executor
    nxt = [0x10000000]

    def fake_alloc(nbytes):
        size = core._Pool._round(nbytes)
        nxt[0] += size
        return nxt[0] - size, size

    monkeypatch.setattr(core.pool, "alloc", fake_alloc)
    monkeypatch.setattr(core.pool, "free", lambda ptr, size: None)
    monkeypatch.setattr(L, "h2d", lambda ptr, arr: None)
    monkeypatch.setitem(executor.flags, "enable_replay", True)
    executor._plans.clear()
    return executor


@pytest.mark.parametrize("groups,by,variable", [(1, "w", "MJT_NO_FASTPATH"), (1, "w", "MJT_MOST_WORKSPACE"), (32, "x", "MJT_NO_FASTPATH")])
def test_replayed_graph_whose_call_is_handed_back_is_worked_out_anew(fake_buffers, monkeypatch, groups, by, variable):
    """A route that was there when the plan was made and is not any more: the graph takes the route without it, as on a first
    execution, replayed by its calls or by recorded launches."""
    stats = fake_buffers.stats

    def step():
        v = {"x": jt.array(np.ones((64, 32, 15, 13), np.float32)), "w": jt.array(np.ones((32, 32 // groups, 3, 3), np.float32))}
        g = jt.array(np.ones((64, 32, 15, 13), np.float32))
        y = jt.nn.conv2d(v["x"], v["w"], padding=1, groups=groups)
        out = jt.grad((y * g).sum(), v[by])
        jt.sync([out])
        return out

    for warm in (2, 4):
        for _ in range(warm):
            step()
        before = dict(stats)
        monkeypatch.setenv(variable, "1")
        assert step()._buf is not None
        assert stats["plans"] == before["plans"] + 1 and stats["replays"] == before["replays"]
        step()
        assert stats["replays"] == before["replays"] + 1
        monkeypatch.delenv(variable)
        fake_buffers._plans.clear()


def test_replay_that_fails_leaves_its_results_uncomputed(fake_buffers):
    """An error in the middle of a replay: the results have no buffer that would pass for computed, and the next attempt computes them."""
    def graph():
        x = jt.array(np.ones((64, 48), np.float32))
        return [x.sum([0]), (x * x).sum([1])]

    for _ in range(2):
        jt.sync(graph())
    plan = next(iter(fake_buffers._plans.values()))
    outs = graph()
    plan.calls.append((lambda: L.ERR_UNSUPPORTED - 1, ()))             # some other error
    plan.native = False
    with pytest.raises(L.MjtError):
        jt.sync(outs)
    assert all(v._buf is None and v._op is not None for v in outs)
    plan.calls.pop()
    jt.sync(outs)
    assert all(v._buf is not None and v._op is None for v in outs)


@pytest.mark.parametrize("shared_first", [True, False])
@pytest.mark.parametrize("twice", [False, True])
def test_replayed_result_is_the_memory_of_its_own_input(fake_buffers, shared_first, twice):
    """A reshape of one input, replayed after an execution in which the two inputs were one buffer (and the other way round): the
    result is that input's memory, not the other's."""
    def step(shared):
        a = jt.array(np.ones((8, 4), np.float32)) + 1.0
        b = a.reshape([32]) if shared else jt.array(np.ones(32, np.float32)) + 2.0
        jt.sync([a])
        jt.sync([b])
        assert (b._buf is a._buf) == shared
        y, z = b.reshape([4, 8]), a * 2.0
        if twice:
            y = y.reshape([2, 16])
        jt.sync([y, z])
        return b, y

    for shared in (shared_first, shared_first, not shared_first, not shared_first, shared_first):
        replays = fake_buffers.stats["replays"]
        b, y = step(shared)
        assert y._buf is b._buf
    assert fake_buffers.stats["replays"] > replays + 1


@pytest.mark.parametrize("targets", ["x1 x2 w1 w2", "w1 w2 x1 x2", "w2 x1 x2 w1", "x2 w1 x1 w2", "x1 w2 x2", "w1 x2 w2"])
@pytest.mark.parametrize("shared,branches", [(False, 2), (True, 2), (False, 3)])
@pytest.mark.parametrize("pairs", [True, False])
def test_depthwise_branches_that_are_summed(fake_buffers, monkeypatch, targets, shared, branches, pairs):
    """Branches that are summed send one dy to several input and weight gradients: each is computed, by one call, and no more calls
    make two at once than there are of either (none without the flag)."""
    monkeypatch.setitem(fake_buffers.flags, "enable_gradient_pairs", pairs)
    v = {}
    for i in range(1, branches + 1):
        v["x%d" % i] = v["x1"] if shared and i > 1 else jt.array(np.ones((8, 32, 14, 14), np.float32)) * float(i)
        v["w%d" % i] = jt.array(np.ones((32, 1, 3, 3), np.float32)) * float(i)
    jt.sync(list(v.values()))
    fake_buffers._plans.clear()
    y = sum((jt.nn.conv2d(v["x%d" % i], v["w%d" % i], padding=1, groups=32) for i in range(2, branches + 1)), jt.nn.conv2d(v["x1"], v["w1"], padding=1, groups=32))
    names = [n for n in targets.split() if not (shared and n == "x2")] + (["x3", "w3"] if branches == 3 else [])
    grads = jt.grad((y * y).sum(), [v[n] for n in names])
    jt.sync(grads)
    assert all(g._buf is not None for g in grads)
    plan, = fake_buffers._plans.values()
    made, both = [], 0
    for fn, args in plan.calls:
        outs = {"mjt_conv2d_meta_backward_depthwise": (3, 4), "mjt_conv2d_meta_dgrad_depthwise": (2,), "mjt_conv2d_meta_wgrad_grouped": (2,)}.get(fn.__name__, ())
        made += [args[k]._obj.ptr for k in outs]
        both += len(outs) == 2
    n_x, n_w = sum(n[0] == "x" for n in names) * (branches if shared else 1), sum(n[0] == "w" for n in names)
    assert len(made) == len(set(made)) == n_x + n_w and both == (min(n_x, n_w) if pairs else 0)
    if not shared:
        assert set(made) == {g._buf.ptr for g in grads}


@pytest.mark.parametrize("zeros", [(0.0, 0.0), (0, 0), (False, 0.0), "arrays", "arrays of halves"])
def test_masks_read_from_results_are_replayed(fake_buffers, zeros):
    """convolution, select against zero, convolution, with gradients: whatever the zeros are, the mask is read from the select's result and
    the graph is replayed and recorded."""
    stats = fake_buffers.stats
    w1, w2 = jt.array(np.ones((8, 4, 3, 3), np.float32)), jt.array(np.ones((8, 8, 3, 3), np.float32))
    x = jt.array(np.ones((2, 4, 9, 9), np.float32))
    jt.sync([x, w1, w2])
    fake_buffers._plans.clear()

    def step():
        zero = [jt.array(np.zeros([1], np.float16 if "halves" in zeros else np.float32)) for _ in range(2)] if isinstance(zeros, str) else zeros
        v = jt.nn.conv2d(x, w1, padding=1)
        z = jt.nn.conv2d(jt.ternary(v > zero[0], v, zero[1]), w2, padding=1)
        jt.sync([z] + list(jt.grad((z * z).sum(), [w1, w2])))
    before = dict(stats)
    for _ in range(4):
        step()
    assert stats["plans"] == before["plans"] + 1 and stats["replays"] == before["replays"] + 3
    assert stats["recorded_launches"] > before["recorded_launches"]
    assert stats["fused_products"] == before["fused_products"] + 8          # the select behind one product, the mask behind another


def test_fused_rows_descriptor_is_checked(compile_only):
    """mjt_fused_rows: what it hands back runs part by part, what makes no sense is an error; nothing is launched."""
    L, lib = compile_only, compile_only.load()
    f32, P = L.DTYPE_CODE["float32"], 0x1000

    def call(shape, n_row, mask=0, reduce_op="add", dtype=f32, in_space=1, second_in=1):
        fv = [L.FusedVar(L.VAR_INPUT, dtype, P, 0, 0, 0, 0), L.FusedVar(L.VAR_INTERMEDIATE, dtype, None, 0, 0, 0, in_space),
              L.FusedVar(L.VAR_INPUT, dtype, P, 0, 0, mask, 0), L.FusedVar(L.VAR_OUTPUT, dtype, P, 0, 0, 0, 0)]
        fo = [L.FusedOp(L.FOP_ROW_REDUCE, L.OP_CODE[reduce_op], (0, 0, 0), 1), L.FusedOp(L.FOP_BINARY, L.OP_CODE["divide"], (2, second_in, 0), 3)]
        d = L.FusedDesc(len(shape), tuple(shape), 4, (L.FusedVar * 4)(*fv), 2, (L.FusedOp * 2)(*fo))
        return lib.mjt_fused_rows(ctypes.byref(d), n_row)
    assert call((100, 512), 1) == 0 and call((7, 9, 30, 20), 2) == 0 and call((5, 16384), 1, reduce_op="maximum") == 0
    assert call((100, 512), 1, mask=0b10) == 0 and call((100, 512), 1, mask=0b01) == 0 and call((100, 512), 1, mask=0b11) == 0
    assert call((7, 9, 30, 20), 2, mask=0b1000) == L.ERR_UNSUPPORTED                   # along part of the rows
    assert call((5, 16385), 1) == L.ERR_UNSUPPORTED and call((0, 64), 1) == L.ERR_UNSUPPORTED and call((64, 0), 1) == L.ERR_UNSUPPORTED
    assert call((100, 512), 1, reduce_op="multiply") == L.ERR_UNSUPPORTED and call((100, 512), 1, dtype=L.DTYPE_CODE["int32"]) == L.ERR_UNSUPPORTED
    assert call((100, 512), 0) == L.ERR_INVALID and call((100, 512), 2) == L.ERR_INVALID
    assert call((100, 512), 1, in_space=0) == L.ERR_INVALID and call((100, 512), 1, second_in=9) == L.ERR_INVALID


@pytest.mark.parametrize("column_sum", [False, True])
def test_fused_rows_counts_rows_in_32_bits(compile_only, column_sum):
    """The kernel's row counter goes one step past the last row: 2^20 workgroups of 256 rows, or with column sums the 1024 that 256 compute units
    are given.  Nothing is launched."""
    L, lib = compile_only, compile_only.load()
    f32, P = L.DTYPE_CODE["float32"], 0x1000

    def call(rows):
        fv = [L.FusedVar(L.VAR_INPUT, f32, P), L.FusedVar(L.VAR_INTERMEDIATE, f32, None, 0, 0, 0, 1), L.FusedVar(L.VAR_OUTPUT, f32, P, 0, 0, 0, 0), L.FusedVar(L.VAR_OUTPUT, f32, P, 0, 0, 0, 2)]
        fo = [L.FusedOp(L.FOP_ROW_REDUCE, L.OP_CODE["maximum"], (0, 0, 0), 1), L.FusedOp(L.FOP_BINARY, L.OP_CODE["subtract"], (0, 1, 0), 2), L.FusedOp(L.FOP_COLUMN_SUM, L.OP_CODE["add"], (2, 0, 0), 3)]
        n = 4 if column_sum else 3
        d = L.FusedDesc(2, (rows, 4), n, (L.FusedVar * n)(*fv[:n]), n - 1, (L.FusedOp * (n - 1))(*fo[:n - 1]))
        return lib.mjt_fused_rows(ctypes.byref(d), 1)
    step = 1024 * 256 if column_sum else 2 ** 20 * 256
    assert call(1100000000) == 0 and call(2 ** 31 - step - 1) == 0
    for rows in (2 ** 31 - step, 2 ** 31 - 70000, 2 ** 31, 2 ** 33):
        assert call(rows) == L.ERR_UNSUPPORTED


class _Rows:
    """mjt_fused_rows worked out in numpy from its descriptor; `at` has the arrays in memory by address."""

    def __init__(self):
        self.at, self.calls = {}, 0

    def __call__(self, desc, n_row_axes):
        d = desc._obj
        shape = [d.shape[a] for a in range(d.ndim)]
        rows = int(np.prod(shape[:d.ndim - n_row_axes]))
        cols = int(np.prod(shape)) // rows
        name = {v: k for k, v in L.OP_CODE.items()}
        val, declared = {}, {}
        for i in range(d.n_vars):
            v = d.vars[i]
            declared[i] = v.reserved & 3
            if v.role == L.VAR_SCALAR:
                val[i] = np.float64(v.fvalue)
            elif v.role == L.VAR_INPUT:
                a = self.at[int(v.ptr)]
                val[i] = np.broadcast_to(a.reshape([1 if v.bcast_mask >> q & 1 else shape[q] for q in range(d.ndim)]), shape).reshape(rows, cols)
        for k in range(d.n_ops):
            o = d.ops[k]
            a = [val[o.inp[j]] for j in range(2 if o.kind == L.FOP_BINARY else 1)]
            if o.kind == L.FOP_ROW_REDUCE:
                r = {"add": np.sum, "mean": np.mean, "maximum": np.max}[name[o.op]](a[0], axis=1, keepdims=True)
            elif o.kind == L.FOP_COLUMN_SUM:
                r = a[0].sum(0, keepdims=True)
            elif o.kind == L.FOP_BROADCAST:
                r = a[0]
            elif o.kind == L.FOP_UNARY:
                r = {"sqrt": np.sqrt, "exp": np.exp}[name[o.op]](a[0])
            else:
                r = {"add": np.add, "subtract": np.subtract, "multiply": np.multiply, "divide": np.divide}[name[o.op]](*a)
            if o.kind not in (L.FOP_ROW_REDUCE, L.FOP_COLUMN_SUM):
                r = np.broadcast_to(r, [rows, 1] if declared[o.out] == 1 else [rows, cols]) if declared[o.out] == 0 or np.ndim(r) < 2 else r[:, :1]
            val[o.out] = r
            if d.vars[o.out].role == L.VAR_OUTPUT:
                self.at[int(d.vars[o.out].ptr)] = r
        self.calls += 1
        return 0


@pytest.mark.parametrize("graph,fused", list(zip(rows_graphs.GRAPHS, [0, 0, 0, 0, 1, 1, 1, 1])) + [(None, 1)])
def test_rows_of_square_matrices_are_told_from_their_columns(fake_buffers, monkeypatch, graph, fused):
    """What runs as one kernel over rows where there are as many rows as columns: a value per row that is read per column is read from
    memory, behind the kernel that makes it.  The descriptors are worked out in numpy."""
    rows = _Rows()
    monkeypatch.setitem(fake_buffers.flags, "enable_replay", False)
    rng = np.random.default_rng(3)
    X, E = rng.uniform(0.5, 1.5, (256, 256) if graph else (16, 12, 16, 12)), rng.uniform(0.5, 1.5, 256)
    x, e = jt.array(X.astype(np.float32)), jt.array(E.astype(np.float32))
    jt.sync([x, e])
    outs = graph(x, X, e, E) if graph else rows_graphs.several_axes(x, X)

    def call(desc, n):
        for v, want in [(x, X), (e, E)] + outs:                # what lies in memory when the kernel runs
            if v._buf is not None:
                rows.at.setdefault(v._buf.ptr, want)
        return rows(desc, n)
    monkeypatch.setattr(L.load(), "mjt_fused_rows", call)
    jt.sync([v for v, _ in outs])
    checked = 0
    for v, want in outs:
        got = rows.at.get(v._buf.ptr)
        if got is not None and got is not want:
            checked += 1
            assert np.allclose(got.reshape(want.shape), want, rtol=1e-9)
    assert rows.calls == fused and (checked > 0) == (fused > 0)


def test_native_constructors_take_what_they_took():
    """unary, binary, ternary, broadcast and reduce (csrc/py/graph.cpp): keyword arguments, numbers and arrays as operands, numpy integers and
    negative axes, what is refused and how; a Var's readers, ids and history are kept as the classes' own constructors keep them."""
    import gc
    from jittor_amd import core
    x = jt.array(np.ones((2, 3), np.float32))
    assert jt.binary(x=x, y=2, op="add").shape == [2, 3] and jt.unary(op="sqrt", x=4.0).dtype == "float32" and jt.ternary(cond=x > 0, x=x, y=1.0).shape == [2, 3]
    assert jt.reduce(x, "add", dims=np.int64(-1)).shape == [2] and jt.reduce(x, op="mean", dims=(0, 1), keepdims=True).shape == [1, 1] and x.sum([]).shape == [1]
    assert jt.broadcast(x, (np.int32(4), 2, 3), [0]).shape == [4, 2, 3] and jt.broadcast(x, [2, 3]) is x and jt.broadcast(jt.array([1.0]), shape=x).shape == [2, 3]
    assert jt.binary(np.arange(3), x, "multiply").shape == [2, 3] and (x + True).shape == [2, 3] and jt.unary(x, "float32") is x and jt.unary(x, "float64").dtype == "float64"
    for call, error, text in ((lambda: jt.binary(x, 1, "nope"), ValueError, "unknown binary op 'nope'"), (lambda: jt.unary(x, "nope"), ValueError, "unknown unary op 'nope'"),
                              (lambda: jt.binary(x, jt.array(np.ones((2, 4), np.float32)), "add"), ValueError, r"Shape not match, x:\[2, 3\] y:\[2, 4\]"),
                              (lambda: jt.reduce(x, "add", 2), ValueError, "Wrong dims number"), (lambda: jt.reduce(x, "less"), ValueError, "not associative|unknown"),
                              (lambda: jt.broadcast(x, [4, 2, 3], [5]), ValueError, "Wrong dims number"), (lambda: jt.broadcast(x, [-1, 2, 3]), ValueError, "greater than 0|not match"),
                              (lambda: jt.binary(x, object(), "add"), TypeError, "cannot convert"), (lambda: jt.binary(x, 1), TypeError, "missing"),
                              (lambda: jt.binary(x, 1, "add", 3), TypeError, "at most"), (lambda: jt.binary(x, 1, op="add", z=2), TypeError, "unexpected"),
                              (lambda: jt.broadcast(x, [1] * 12), ValueError, "dims are supported|not match")):
        with pytest.raises(error, match=text):
            call()
    y = x * x
    assert [r() for r in x._consumers][-2:] == [y._op, y._op] and y._history == (y._op, (x, x)) and y._op.out is y and y._op.id < y.id and y._op.amp == 0
    with jt.no_grad():
        assert (x * 2.0)._history is None
    for _ in range(600):
        x + 1.0                                                # dead readers of a long-lived var are dropped now and then
    assert len(x._consumers) < 300
    gc.collect()
    ref = core._ref(y._op)
    del y
    assert ref() is None                                       # no cycle keeps a graph alive
    with jt.flag_scope(compile_options={"k": 3}):
        assert (x + 1.0).compile_options == {"k": 3}


def test_native_front_end_is_this_interpreters():
    """The extension carries the interpreter's tag, so that another one does not load it; where it is missing the import says what to do."""
    import sysconfig
    from jittor_amd import _graph
    assert os.path.basename(_graph.__file__) == "_graph" + sysconfig.get_config_var("EXT_SUFFIX") != "_graph.so"
    code = "import sys; sys.modules['jittor_amd._graph'] = None; import jittor_amd"
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=120)
    assert r.returncode != 0 and "make -C jittor_amd/csrc" in r.stderr, r.stderr[-300:]


def test_native_constructors_that_find_no_common_shape_raise():
    """A select between no elements and one: an error, as in byte code, where the native one ran out of stack.  (In a process of its own.)"""
    code = """if 1:
        import numpy as np
        import jittor_amd as jt
        none, one = jt.array(np.ones([0], np.float32)), jt.array(np.ones([1], np.float32))
        for a in ((none, one, none), (one, none, none), (none, none, one), (none > 0, one, one)):
            try:
                jt.ternary(*a)
            except RecursionError:
                print("refused")
            else:
                print("made")
        """
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.split() == ["refused"] * 4, (r.returncode, r.stdout, r.stderr[-500:])


@pytest.mark.parametrize("dims", ["0", ["0"], [1.0], 1.0, np.float32(1), None, [[1]], [None], np.array(1)])
def test_named_axes_are_integers(dims):
    x = jt.array(np.ones((2, 3), np.float32))
    for call in (lambda: jt.reduce(x, "add", dims), lambda: jt.broadcast(x, [4, 2, 3], dims)):
        with pytest.raises(TypeError):
            call()
    assert jt.reduce(x, "add", [np.int64(1), True]).shape == [2] and jt.reduce(x, "add", np.array([0, -1])).shape == [1] and jt.broadcast(x, [4, 2, 3], range(1)).shape == [4, 2, 3]


def test_element_counts_do_not_wrap_round():
    """Extents whose product passes 2^63 are refused; with an extent of 0 there are no elements whatever the others are."""
    x = jt.array(np.ones([1], np.float32))
    for shape in ([2 ** 40, 2 ** 40], [2 ** 32, 2 ** 31], [2 ** 21] * 3):
        with pytest.raises(OverflowError):
            jt.broadcast(x, shape)
    assert jt.broadcast(x, [2 ** 31, 2 ** 31]).num == 2 ** 62 and jt.broadcast(x, [2 ** 40, 2 ** 40, 0]).num == 0


def test_graph_keys_tell_graphs_apart():
    """What a key depends on: ops, attributes, shapes, types, wiring, which results are asked for, what is computed already, flags, the
    register; the same graph built again has the same key."""
    from jittor_amd import _graph, executor

    def key(build, targets=-1):
        vs = build()
        ts = [vs[targets]] if isinstance(targets, int) else [vs[i] for i in targets]
        return _graph.signature(_graph.pending_ops(ts), ts, executor.flags), vs

    def base(shape=(4, 6), dt="float32", op="add", k=2.0, dims=(1,), swap=False, twice=False, idx="i0"):
        a, b = jt.array(np.ones(shape, np.float32)).cast(dt) if dt != "float32" else jt.array(np.ones(shape, np.float32)), jt.array(np.ones(shape, np.float32))
        c = jt.binary(*((b, a) if swap else (a, a if twice else b)), op)
        d = c * k
        return [a, b, c, d, d.sum(list(dims), keepdims=True), d.reindex([shape[0]], [idx, "0"])]

    seen = {}
    for name, kw, targets in (("base", {}, 4), ("shape", {"shape": (4, 7)}, 4), ("dtype", {"dt": "float64"}, 4), ("op", {"op": "subtract"}, 4), ("dims", {"dims": (0,)}, 4),
                              ("twice", {"twice": True}, 4), ("targets", {}, (3, 4)), ("reindex", {}, 5), ("index", {"idx": "3-i0"}, 5), ("other", {}, 3)):
        k, _ = key(lambda: base(**kw), targets)
        assert k is not None and k not in seen.values(), name
        seen[name] = k
        assert key(lambda: base(**kw), targets)[0] == k
    assert key(lambda: base(k=3.0), 4)[0] == seen["base"]       # a number's value is data
    k0, vs = key(lambda: base(), 4)
    with jt.flag_scope(enable_reduce_fusion=False):
        assert _graph.signature(_graph.pending_ops([vs[4]]), [vs[4]], executor.flags) != k0
    with jt.flag_scope(amp_reg=32):
        assert _graph.signature(_graph.pending_ops([vs[4]]), [vs[4]], executor.flags) != k0
    vs[2].stop_fuse()
    assert _graph.signature(_graph.pending_ops([vs[4]]), [vs[4]], executor.flags) != k0


def test_graph_keys_tell_a_select_against_zero(fake_buffers):
    """What a relu's mask is read from depends on whether the threshold and the other operand are zero: the key of a graph with a select
    tells zeros from other numbers, other numbers are data."""
    from jittor_amd import _graph
    w = jt.array(np.ones((8, 4, 3, 3), np.float32))
    jt.sync([w])

    def step(threshold, other):
        x = jt.array(np.ones((2, 4, 9, 9), np.float32)) * 2.0
        jt.sync([x])
        y = jt.ternary(x > (0.0 if threshold == 0 else jt.array(np.float32([threshold]))), x, jt.array(np.float32([other])))
        z = jt.nn.conv2d(y, w, padding=1)
        gx = jt.grad((z * z).sum(), x)
        key = _graph.signature(_graph.pending_ops([z, gx]), [z, gx], fake_buffers.flags)
        replays = fake_buffers.stats["replays"]
        jt.sync([z, gx])
        return key, fake_buffers.stats["replays"] - replays

    keys = {}
    for threshold, other, known in ((0, 0, 0), (0, 5, 0), (3, 0, 0), (2, 7, 0), (0, 0, 1), (0, 6, 1), (-1, 0, 1), (5, 5, 1)):
        key, replays = step(threshold, other)
        assert replays == known, (threshold, other)
        assert keys.setdefault((threshold == 0, other == 0), key) == key
    assert len(set(keys.values())) == len(keys) == 4
    number = lambda v, dtype: _graph.zero_number(jt.array(np.asarray(v, dtype)))
    assert number([0], np.float32) and number([0], np.int64) and number([False], np.bool_) and number([0], np.float16)
    assert not number([1e-45], np.float32) and not number([-0.0], np.float32) and not number([0, 0], np.float32) and not number([1], np.int8)
    assert not _graph.zero_number(jt.array(np.zeros([1], np.float32)) + 0.0)
