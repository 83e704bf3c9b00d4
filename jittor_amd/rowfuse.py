"""Groups and row reductions that run as one kernel.

The executor partitions a graph into element groups, reduces and the groups that are a reduce's prologue
(executor.py; python/jittor/src/executor.cc:318-555); a normalisation or a softmax becomes a chain of them in which
every link reads the same rows from memory again.  Where all links of such a chain work on one [rows, columns] shape,
mjt_fused_rows runs them together: a row stays in registers between its reductions, column sums (the gradients of a
scale and a shift) ride along.  What runs together is chosen when a graph is executed for the first time; replays
issue the recorded calls.
"""
import ctypes
import heapq

from . import _lib
from .core import UnaryOp, BinaryOp, TernaryOp, BroadcastOp, ReduceOp

MOST_COLUMNS = 16384             # a row has to fit the registers of a workgroup (csrc/op_rows.cpp)
MOST_OPS = 128
# A small space is bound by its launches, 3 us each, not by its memory: a training step's chain of many is worth a kernel of its own, the
# three of a normalisation, whose kernels many graphs share, are not (us a pass, apart / as one: softmax 307 x 69 with its gradient, seven
# launches, 79 / 46; layer normalisation with its gradients float32 40 x 500 126 / 80, bfloat16 27 x 1092 161 / 106; a small CNN step with a
# cross entropy over 4 x 5 310 / 277).
SMALL, SMALL_PARTS = 1 << 15, 6
FULL, ROW, COLUMN, ROUNDED = 0, 1, 2, 256
SINGLE, OTHER = 3, 4
_SUMMED = ("float32", "float16", "bfloat16")


class Task:
    """One step of an execution: an element group, a reduce (with its prologue group), or anything else."""
    __slots__ = ("run", "members", "reduce", "reads", "writes", "place", "narrowed", "node")

    def __init__(self, run, reads, writes, members=(), reduce=None, node=None):
        self.run, self.members, self.reduce, self.node = run, list(members), reduce, node
        self.reads, self.writes = reads, writes                # ids of the vars in memory that it needs and leaves
        self.place, self.narrowed = None, None                 # narrowed: the var a column sum is cast to, instead of its own


def _space(mask, shape, first):
    """What a tensor read through a broadcast mask is to a [rows, columns] space: full, one value per row, per column, or one."""
    lead = [bool(mask >> a & 1) for a in range(first) if shape[a] != 1]
    tail = [bool(mask >> a & 1) for a in range(first, len(shape)) if shape[a] != 1]
    if not any(lead) and not any(tail):
        return FULL
    if not any(lead) and all(tail):
        return ROW
    if all(lead) and not any(tail):
        return COLUMN
    return SINGLE if all(lead) and all(tail) else OTHER


def _number(u):
    return u._op is None and u._host is not None and u.num == 1


def _row_shaped(shape, full, first):
    return shape[:first] == full[:first] and all(n == 1 for n in shape[first:])


class _Chooser:
    def __init__(self, tasks, ins, pre):
        self.tasks, self.ins, self.pre = tasks, ins, pre

    def place_of(self, t, full, first, row_values):
        """FULL (an element group or a row reduce over `full`), ROW (a group of one value per row), COLUMN (a sum over the rows), or None.
        `row_values`: the vars that tasks ahead of this one make as one value per row.  Where there are as many rows as columns a
        broadcast can read them per column too: that takes other rows' values, which are complete when the kernel ends."""
        members, red = t.members, t.reduce
        if not members and red is None:
            return None
        if red is not None:
            x = red.inputs[0]
            nd = len(full)
            if list(x.shape) != full or x.dtype not in _SUMMED or red.out.dtype not in _SUMMED or getattr(x, "_stop_fuse", False):
                return None
            tail = ((1 << nd) - 1) >> first << first
            if red.reduce_mask == tail:
                if red.op not in ("add", "mean", "maximum", "minimum"):
                    return None
            elif red.reduce_mask != (1 << first) - 1 or red.op != "add":
                return None
            if getattr(red.out, "_stop_fuse", False):
                return None
        if members:
            shape = list(members[-1].out.shape)
            rowwise = red is None and shape != full and _row_shaped(shape, full, first)
            if shape != full and not rowwise:
                return None
            for op in members:
                if getattr(op.out, "_stop_fuse", False) or not isinstance(op, (UnaryOp, BinaryOp, TernaryOp, BroadcastOp)):
                    return None
                if isinstance(op, BroadcastOp):
                    mask = op.bcast_mask & ((1 << len(shape)) - 1)
                    reads = self.ins(op)
                    if any(getattr(u, "_stop_fuse", False) for u in reads):
                        return None
                    if all(_number(u) for u in reads):
                        continue
                    sp = _space(mask, shape, min(first, len(shape)))
                    if sp == OTHER or (rowwise and sp not in (FULL, SINGLE)):
                        return None
                    if sp != (FULL if rowwise else ROW) and any(u.id in row_values for u in reads):
                        return None
                else:
                    for u in op.inputs:
                        if getattr(u, "_stop_fuse", False) or not (list(u.shape) == shape or _number(u)):
                            return None
            if rowwise:
                return ROW
        return COLUMN if red is not None and red.reduce_mask == (1 << first) - 1 else FULL

    def shapes(self):
        """The [rows, columns] spaces that some row reduce of the graph works on, largest first."""
        found = {}
        for t in self.tasks:
            red = t.reduce
            if red is None:
                continue
            shape = list(red.inputs[0].shape)
            nd, n = len(shape), bin(red.reduce_mask).count("1")
            first = nd - n
            if n < 1 or first < 1 or red.reduce_mask != ((1 << nd) - 1) >> first << first:
                continue
            cols = 1
            for k in shape[first:]:
                cols *= k
            num = red.inputs[0].num
            if 0 < cols <= MOST_COLUMNS and num > 0:
                found[(tuple(shape), first)] = num
        return sorted(found, key=lambda k: -found[k])

    def cluster(self, full, first):
        """Tasks that can run as one: no path from one of them to another leaves them.  The first part of them, connected by the
        full-size vars they share, that is worth it."""
        full = list(full)
        num = 1
        for k in full:
            num *= k
        writer = {v: i for i, t in enumerate(self.tasks) for v in t.writes}
        # vars that some group over the full shape reads as one value per column
        by_column = {u.id for t in self.tasks for op in t.members if isinstance(op, BroadcastOp) and list(op.out.shape) == full
                     and _space(op.bcast_mask & ((1 << len(full)) - 1), full, first) == COLUMN for u in self.ins(op)}
        behind, inside, place, row_values = set(), set(), {}, set()
        for i, t in enumerate(self.tasks):
            deps = {writer[v] for v in t.reads if v in writer and writer[v] != i}
            place[i] = None if deps & behind else self.place_of(t, full, first, row_values)
            if place[i] == ROW and not deps & inside and by_column & t.writes:
                place[i] = None                                # as many rows as columns: it runs ahead, for all its readers
            if place[i] is not None:
                inside.add(i)
                if place[i] == COLUMN:                         # complete when the kernel ends
                    behind.add(i)
                elif place[i] == ROW:
                    row_values |= t.writes
                elif t.reduce is not None:
                    row_values.add(t.reduce.out.id)
            elif deps & (inside | behind):
                behind.add(i)
        # connected parts
        parent = {i: i for i in inside}

        def find(a):
            while parent[a] != a:
                parent[a] = parent[parent[a]]
                a = parent[a]
            return a
        size = {}
        for t in self.tasks:
            for op in t.members:
                for u in self.ins(op):
                    size[u.id] = u.num
            if t.reduce is not None:
                size[t.reduce.inputs[0].id] = t.reduce.inputs[0].num
        at = {}
        for i in sorted(inside):
            for v in list(self.tasks[i].reads) + list(self.tasks[i].writes):
                if v in at and (size.get(v) == num or writer.get(v) in inside):
                    parent[find(i)] = find(at[v])
                at.setdefault(v, i)
        parts = {}
        for i in sorted(inside):
            parts.setdefault(find(i), []).append(i)
        for part in parts.values():
            n_rows = sum(1 for i in part if self.tasks[i].reduce is not None and place[i] == FULL)
            n_ops = sum(len(self.tasks[i].members) + 1 for i in part)
            passes = sum(1 for i in part if place[i] != ROW)   # over the full size, which become one
            if n_rows and (passes >= 2 if num >= SMALL else len(part) >= SMALL_PARTS) and n_ops <= MOST_OPS:
                for i in part:
                    self.tasks[i].place = place[i]
                return part
        return None


def merge(tasks, ins, pre, consumers, target_ids, ex):
    """The tasks with clusters of them replaced by one task each, in an order in which every task finds what it reads."""
    done = False
    refused = set()
    while True:
        ch = _Chooser(tasks, ins, pre)
        for full, first in ch.shapes():
            if (full, first, len(tasks)) in refused:
                continue
            part = ch.cluster(full, first)
            if part is None:
                refused.add((full, first, len(tasks)))
                continue
            inner = [tasks[i] for i in part]
            casts = []
            for t in inner:
                t.narrowed = None
                users = consumers.get(t.reduce.out.id, ()) if t.place == COLUMN else ()
                if len(users) == 1 and t.reduce.out.id not in target_ids and isinstance(users[0], UnaryOp) and users[0].op == "cast" \
                        and users[0].out.dtype in _SUMMED and not getattr(users[0].out, "_stop_fuse", False):
                    alone = [q for q in tasks if q.reduce is None and q.members == [users[0]]]
                    if alone:                                  # the sum is stored in the type it is cast to
                        t.narrowed = users[0].out
                        casts.append(alone[0])
            writes = set().union(*(t.writes for t in inner + casts))
            reads = set().union(*(t.reads for t in inner)) - writes
            one = Task(_runner(inner, casts, list(full), first, ins, pre, consumers, target_ids, ex), reads, writes)
            gone = {id(t) for t in inner + casts}
            tasks = _ordered([t for t in tasks if id(t) not in gone] + [one], {id(one): part[-1]}, tasks)
            done = True
            break
        else:
            return tasks if done else None


def _ordered(tasks, where, before):
    """Topological order that keeps to the order the tasks had."""
    index = {id(t): i for i, t in enumerate(before)}
    index.update(where)
    writer = {v: t for t in tasks for v in t.writes}
    waits, after = {}, {}
    for t in tasks:
        deps = {id(writer[v]): writer[v] for v in t.reads if v in writer and writer[v] is not t}
        waits[id(t)] = len(deps)
        for d in deps:
            after.setdefault(d, []).append(t)
    heap = [(index[id(t)], k, t) for k, t in enumerate(tasks) if not waits[id(t)]]
    heapq.heapify(heap)
    out, k = [], len(tasks)
    while heap:
        _, _, t = heapq.heappop(heap)
        out.append(t)
        for q in after.get(id(t), ()):
            waits[id(q)] -= 1
            if not waits[id(q)]:
                k += 1
                heapq.heappush(heap, (index[id(q)], k, q))
    assert len(out) == len(tasks)
    return out


def _runner(inner, casts, full, first, ins, pre, consumers, target_ids, ex):
    def run():
        if not run_rows(inner, full, first, ins, pre, consumers, target_ids, ex):
            for t in inner + casts:
                t.run()
    return run


def run_rows(inner, full, first, ins, pre, consumers, target_ids, ex):
    """One mjt_fused_rows for the tasks; False where the library does not take them."""
    cap = ex._cap
    lib = ex._libh()
    nodes = {op.id for t in inner for op in t.members} | {t.reduce.id for t in inner if t.reduce is not None}
    fvars, fops, prov, made, read = [], [], [], {}, {}

    def add_var(role, dtype, ptr=None, mask=0, reserved=0, scalar=None):
        fv = _lib.FusedVar()
        fv.role, fv.dtype, fv.ptr, fv.bcast_mask, fv.reserved = role, _lib.DTYPE_CODE[dtype], ptr, mask, reserved
        if scalar is not None:
            fv.fvalue, fv.ivalue = ex._scalar_value(scalar)
        fvars.append(fv)
        if cap is not None:                                    # where the pointer / the value came from, for replays
            if scalar is not None:
                prov.append((len(fvars) - 1, scalar, None))
            elif ptr is not None:
                prov.append((len(fvars) - 1, ptr.var, ptr.off))
        return len(fvars) - 1

    space_of = []                                              # of every var, in step with fvars

    def var(space, *a, **kw):
        i = add_var(*a, **kw)
        space_of.append(space)
        return i

    def external(u, mask):
        """A var that is not made here, read through a mask over the full shape."""
        if u.id in made:
            return made[u.id]
        key = (u.id, mask)
        if key not in read:
            if _number(u):
                read[key] = var(SINGLE, _lib.VAR_SCALAR, u.dtype, scalar=u)
            else:
                read[key] = var(_space(mask, full, first), _lib.VAR_INPUT, u.dtype, ptr=ex._ptr_of(u), mask=mask)
        return read[key]

    def add_op(op, in_vars, out_var):
        fo = _lib.FusedOp()
        if isinstance(op, UnaryOp):
            fo.kind, fo.op = _lib.FOP_UNARY, _lib.OP_CODE[op.op]
        elif isinstance(op, BinaryOp):
            fo.kind, fo.op = _lib.FOP_BINARY, _lib.OP_CODE[op.op]
        elif isinstance(op, TernaryOp):
            fo.kind = _lib.FOP_TERNARY
        elif isinstance(op, ReduceOp):
            fo.kind = _lib.FOP_ROW_REDUCE if space_of[out_var] == ROW else _lib.FOP_COLUMN_SUM
            fo.op = _lib.OP_CODE[op.op]
        else:
            fo.kind = _lib.FOP_BROADCAST
        for j, v in enumerate(in_vars):
            fo.inp[j] = v
        fo.out = out_var
        fops.append(fo)
        return out_var

    def result(out, space, own_ids):
        """The var of an op's result: stored where something outside reads it, of its own dtype where another part here does."""
        users = consumers.get(out.id, ())
        if out.id in target_ids or any(c.id not in nodes for c in users):
            i = var(space, _lib.VAR_OUTPUT, out.dtype, ptr=ex._alloc_out(out), reserved=space)
        else:
            rounded = ROUNDED if any(c.id not in own_ids for c in users) else 0
            i = var(space, _lib.VAR_INTERMEDIATE, out.dtype, reserved=space | rounded)
        return i

    tail = ((1 << len(full)) - 1) >> first << first
    for t in inner:
        own = {op.id for op in t.members}
        shape = list(t.members[-1].out.shape) if t.members else full
        whole = (1 << len(shape)) - 1
        for op in t.members:
            if isinstance(op, BroadcastOp):
                mask = op.bcast_mask & whole
                if t.place == ROW:
                    mask = mask | tail                         # a value for all rows, or one per row
                if pre and op.id in pre:
                    # the ops in front of the broadcast: once per row where they read nothing else, per element otherwise
                    local = {}
                    for q in pre[op.id]:
                        qin = [local[u.id] if u.id in local else external(u, mask) for u in q.inputs]
                        sp = ROW if all(space_of[i] in (ROW, SINGLE) for i in qin) and any(space_of[i] == ROW for i in qin) else FULL
                        if t.place == ROW:
                            sp = ROW
                        local[q.out.id] = add_op(q, qin, var(sp, _lib.VAR_INTERMEDIATE, q.out.dtype, reserved=sp))
                    in_vars = [local[op.inputs[0].id]]
                else:
                    in_vars = [external(op.inputs[0], mask)]
            else:
                in_vars = [external(u, tail if t.place == ROW else 0) for u in op.inputs]
            made[op.out.id] = add_op(op, in_vars, result(op.out, ROW if t.place == ROW else FULL, own))
        if t.reduce is not None:
            x = t.reduce.inputs[0]
            made_sum = add_op(t.reduce, [external(x, 0)], _reduced(t, result, var, ex))
            if t.place != COLUMN:
                made[t.reduce.out.id] = made_sum
    desc = _lib.FusedDesc()
    desc.ndim = len(full)
    for i, s in enumerate(full):
        desc.shape[i] = s
    varr, oarr = (_lib.FusedVar * len(fvars))(*fvars), (_lib.FusedOp * len(fops))(*fops)
    desc.n_vars, desc.vars, desc.n_ops, desc.ops = len(fvars), varr, len(fops), oarr
    rc = lib.mjt_fused_rows(ctypes.byref(desc), len(full) - first)
    if rc == _lib.ERR_UNSUPPORTED:
        return False
    _lib.check(rc)
    if cap is not None:
        for i, v, off in prov:
            if off is None:
                cap.scalars.append((varr, i, v))
            else:
                cap.ptrs.append((varr, i, v, off))
    ex.stats["launches"] += 1
    ex.stats["fused_rows"] += 1
    return True


def _reduced(t, result, var, ex):
    out = t.narrowed or t.reduce.out
    if t.place == COLUMN:
        return var(COLUMN, _lib.VAR_OUTPUT, out.dtype, ptr=ex._alloc_out(out), reserved=COLUMN)
    return result(out, ROW, ())
