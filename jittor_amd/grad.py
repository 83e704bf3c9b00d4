"""Reverse-mode gradients of the meta-operator path.

The gradient of every op on this path is again built from ops of the path, as
in the reference: ReindexOp -> reindex_reduce(add)
(python/jittor/src/ops/reindex_op.cc:76-80), ReindexReduceOp -> reindex
(+ an equality mask for maximum / minimum, ops/reindex_reduce_op.cc:45-63),
ReduceOp -> broadcast (ops/reduce_op.cc:339-362), BroadcastToOp -> reduce(add)
(ops/broadcast_to_op.cc:112-117), and the element-wise rules of
ops/binary_op.cc:491-561, ops/unary_op.cc:891-1019, ops/ternary_op.cc:49-56.
The driver follows python/jittor/src/grad.cc:85-284: only float vars carry
gradients, contributions of several consumers are added, a target the loss
does not depend on gets zeros.
"""
from . import _graph
from . import core
from .core import (Var, UnaryOp, BinaryOp, ReduceOp, ReindexOp, ReindexReduceOp,
                   unary, binary, ternary, make_number, reindex, reindex_reduce, array)


# The gradients of cast, negative, exp, log, sqrt, sigmoid, of the four arithmetic ops, of ternary and broadcast and of the reduces add, mean,
# maximum and minimum are in csrc/py/graph.cpp.
def _unary_grad(op, x, y, dout):
    """ops/unary_op.cc:891-1019 (y is the op's output; x is a float)."""
    ns = op.op
    one = lambda: make_number(1, x)
    if ns == "abs":
        return ternary(binary(x, make_number(0, x), "greater_equal"), dout, unary(dout, "negative"))
    if ns == "sin":
        return binary(dout, unary(x, "cos"), "multiply")
    if ns == "cos":
        return binary(dout, unary(unary(x, "sin"), "negative"), "multiply")
    if ns == "tan":
        c = unary(x, "cos")
        return binary(dout, binary(c, c, "multiply"), "divide")
    if ns == "asin":
        return binary(dout, unary(binary(one(), binary(x, x, "multiply"), "subtract"), "sqrt"), "divide")
    if ns == "acos":
        return unary(binary(dout, unary(binary(one(), binary(x, x, "multiply"), "subtract"), "sqrt"), "divide"), "negative")
    if ns == "atan":
        return binary(dout, binary(one(), binary(x, x, "multiply"), "add"), "divide")
    if ns == "sinh":
        return binary(dout, unary(x, "cosh"), "multiply")
    if ns == "cosh":
        return binary(dout, unary(x, "sinh"), "multiply")
    if ns == "tanh":
        c = unary(x, "cosh")
        return binary(dout, binary(c, c, "multiply"), "divide")
    if ns == "asinh":
        return binary(dout, unary(binary(binary(x, x, "multiply"), one(), "add"), "sqrt"), "divide")
    if ns == "acosh":
        return binary(dout, unary(binary(binary(x, x, "multiply"), one(), "subtract"), "sqrt"), "divide")
    if ns == "atanh":
        return binary(dout, binary(one(), binary(x, x, "multiply"), "subtract"), "divide")
    if ns == "erf":
        r = unary(unary(binary(x, x, "multiply"), "negative"), "exp")
        return binary(dout, binary(r, make_number(2 / 1.7724538509055159, x), "multiply"), "multiply")
    if ns == "erfinv":
        r = unary(binary(y, y, "multiply"), "exp")
        return binary(dout, binary(r, make_number(1.7724538509055159 / 2, x), "multiply"), "multiply")
    return None      # round / floor / ceil / logical ops: no gradient


def _binary_grad(op, x, y, z, dout, index):
    """ops/binary_op.cc:491-561 (z is the op's output)."""
    ns = op.op
    if ns == "mod":
        if index == 0:
            return dout
        return unary(unary(binary(x, y, "divide"), "floor"), "negative")
    if ns in ("maximum", "minimum"):
        zeros = make_number(0, dout)
        cond = binary(y, z, "equal")
        return ternary(cond, dout, zeros) if index == 1 else ternary(cond, zeros, dout)
    if ns == "pow":
        if index == 0:
            d = binary(dout, y, "multiply")
            y_1 = binary(y, array(1), "subtract")
            return binary(d, binary(x, y_1, "pow"), "multiply")
        return binary(dout, binary(z, unary(x, "log"), "multiply"), "multiply")
    return None      # comparisons, logical and bitwise ops, floor_divide


def _op_grad(op, inputs, out, dout, index):
    x = inputs[index]
    if isinstance(op, UnaryOp):
        return _unary_grad(op, inputs[0], out, dout)
    if isinstance(op, BinaryOp):
        return _binary_grad(op, inputs[0], inputs[1], out, dout, index)
    if isinstance(op, ReduceOp):                        # ops/reduce_op.cc:339-362
        if op.op == "multiply":
            return binary(core._broadcast_mask(binary(dout, out, "multiply"), x.shape, op.reduce_mask, op.keepdims_mask), x, "divide")
        return None
    if isinstance(op, ReindexOp):                       # ops/reindex_op.cc:76-80: no gradient for the extras
        if index:
            return None
        if getattr(op, "same_memory", False):           # a reshape: its gradient is the reshape back (ops/reshape_op.cc),
            from . import misc                          # which shares dout's buffer, instead of a scatter with atomics
            return misc.reshape(dout, list(x.shape))
        return reindex_reduce(dout, "add", x.shape, op.indexes, op.overflow_conditions, inputs[1:])
    if isinstance(op, ReindexReduceOp):                 # ops/reindex_reduce_op.cc:45-63
        if index:
            return None
        back = lambda v: reindex(v, x.shape, op.indexes, 0, op.overflow_conditions, inputs[1:])
        if op.op in ("add", "void"):                    # void (plain assignment, setitem_op.cc: the gradient of the value is the
            return back(dout)                           # gradient read back where it was written)
        if op.op == "multiply":
            return binary(back(binary(dout, out, "multiply")), x, "divide")
        if op.op in ("maximum", "minimum"):
            cond = binary(x, back(out), "equal")
            return ternary(cond, back(dout), make_number(0, x))
        return None
    return None


def grad(loss, targets, retain_graph=True):
    """jt.grad(loss, targets): list of d loss / d target (grad.cc:85-284).  The seed is ones of the
    loss's shape, so a non-scalar loss is summed implicitly, as in the reference."""
    single = isinstance(targets, Var)
    targets = [targets] if single else list(targets)
    if not loss.is_float():
        raise ValueError("Loss should be float")
    for t in targets:
        if not t.is_float():
            raise ValueError("Targets of grad should be float")

    # the walk, and the gradients of the common ops, are native (csrc/py/graph.cpp); the others are _op_grad's
    out = _graph.gradients(loss, targets, _op_grad)
    return out[0] if single else out
