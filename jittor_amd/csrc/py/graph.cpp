// jittor_amd._graph: what the front end does for every op of every step -- making Vars and ops (core.py), collecting the pending ops
// behind a request and describing them as a key (executor.py), the walk that builds a gradient graph (grad.py) -- on the Python objects themselves, through the interpreter's C interface.
//
// Var and the op classes stay Python classes with the same attributes; this file only fills their instance dictionaries without
// running byte code.  The constructors restate the reference's (python/jittor/src/ops/binary_op.cc:421-474, unary_op.cc:860-889,
// ternary_op.cc:21-47, broadcast_to_op.cc:23-168, reduce_op.cc:257-337, op_utils.cc:19-36).
//
// Why: a training step of a small network was host work, 3.4 us for a Var and its op in byte code (us of host time a step, in byte code /
// here: a small CNN, 79 ops, 582 / 304, of it building its graph and gradient graph 287 / 96; layer normalisation, 40 ops, 248 / 76; a chain
// of 12 element ops 58 / 22).
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <string>
#include <unordered_map>
#include <unordered_set>
#include <vector>

namespace {

constexpr int MOST = 32;                 // extents looked at; Vars have at most g_max_dim

// owned reference
struct Ref {
    PyObject* p;
    Ref(PyObject* q = nullptr) : p(q) {}
    Ref(const Ref&) = delete;
    Ref(Ref&& o) : p(o.p) { o.p = nullptr; }
    Ref& operator=(Ref&& o) { PyObject* old = p; p = o.p; o.p = nullptr; Py_XDECREF(old); return *this; }
    ~Ref() { Py_XDECREF(p); }
    explicit operator bool() const { return p != nullptr; }
    PyObject* give() { PyObject* q = p; p = nullptr; return q; }
};
PyObject* keep(PyObject* p) { Py_XINCREF(p); return p; }

#define NAMES(X) X(shape) X(num) X(dtype) X(_op) X(_history) X(id) X(_out_ref) X(inputs) X(amp) X(op) X(bcast_mask) X(keepdims_mask) X(reduce_mask) X(is_scalar) \
    X(_consumers) X(_compile_options) X(compile_options) X(amp_reg) X(_buf) X(_host) X(_stop_fuse) X(indexes) X(overflow_value) X(overflow_conditions) X(same_memory) X(sig) \
    X(_binary_dtypes) X(binary_dtype_infer) X(unary_dtype_infer) X(reduce_dtype_infer) X(dtype_infer) X(cast) X(add) X(mean) X(float16) X(bfloat16) X(float32)
#define DECLARE(n) PyObject* s_##n;
NAMES(DECLARE)
#undef DECLARE
PyObject* s_void;

// handed over by core.py
PyTypeObject *t_var, *t_unary, *t_binary, *t_ternary, *t_broadcast, *t_reduce, *t_reindex, *t_reindex_reduce;
PyObject *g_flags, *g_dt, *g_grad_enabled, *g_array, *g_as_var, *g_scalars, *g_dtypes, *g_unary_ops, *g_binary_ops, *g_reduce_ops;
long long g_max_dim = 10;
long long g_next_id = 1;

bool is_var(PyObject* o) { return PyObject_TypeCheck(o, t_var); }

PyObject* dict_of(PyObject* o) {
    PyObject** dp = _PyObject_GetDictPtr(o);
    return dp ? *dp : nullptr;
}
// an attribute from the instance (borrowed), null where it is not there
PyObject* own(PyObject* o, PyObject* name) {
    PyObject* d = dict_of(o);
    return d ? PyDict_GetItemWithError(d, name) : nullptr;
}
// an attribute from the instance or its class
Ref attr(PyObject* o, PyObject* name) {
    if (PyObject* v = own(o, name)) return Ref(keep(v));
    if (PyErr_Occurred()) return Ref();
    return Ref(PyObject_GetAttr(o, name));
}
// what most instances leave at the class's None / False
bool absent(PyObject* o, PyObject* name) {
    PyObject* v = own(o, name);
    return !v || v == Py_None;
}
bool flag(PyObject* o, PyObject* name) {
    PyObject* v = own(o, name);
    return v && PyObject_IsTrue(v) == 1;
}
int amp_now(long long* out) {
    PyObject* v = PyDict_GetItemWithError(PyModule_GetDict(g_dt), s_amp_reg);
    if (!v) return -1;
    *out = PyLong_AsLongLong(v);
    return *out == -1 && PyErr_Occurred() ? -1 : 0;
}

struct Shape {
    int n = 0;
    long long e[MOST];
    bool operator==(const Shape& o) const { return n == o.n && !memcmp(e, o.e, sizeof(long long) * n); }
};
bool read_shape(PyObject* seq, Shape* s) {
    Ref f(PySequence_Fast(seq, "a shape is a sequence of integers"));
    if (!f) return false;
    const Py_ssize_t n = PySequence_Fast_GET_SIZE(f.p);
    if (n > MOST) { PyErr_Format(PyExc_ValueError, "at most %lld dims are supported", g_max_dim); return false; }
    s->n = (int)n;
    for (Py_ssize_t i = 0; i < n; i++) {
        PyObject* v = PySequence_Fast_GET_ITEM(f.p, i);
        if (PyLong_Check(v)) {
            s->e[i] = PyLong_AsLongLong(v);
        } else {                                               // int(v): numpy integers, floats
            Ref q(PyNumber_Long(v));
            if (!q) return false;
            s->e[i] = PyLong_AsLongLong(q.p);
        }
        if (s->e[i] == -1 && PyErr_Occurred()) return false;
    }
    return true;
}
bool count_elements(const Shape& s, long long* num) {
    *num = 1;
    bool over = false;
    for (int i = 0; i < s.n; i++) {
        if (s.e[i] == 0) { *num = 0; return true; }
        over = over || __builtin_mul_overflow(*num, s.e[i], num);
    }
    if (over) PyErr_SetString(PyExc_OverflowError, "a shape of 2^63 elements or more");
    return !over;
}
// named axes: an integer or integers
bool read_dims(PyObject* dims, Shape* s) {
    if (PyIndex_Check(dims) && !PySequence_Check(dims)) {
        s->n = 1;
        s->e[0] = PyNumber_AsSsize_t(dims, PyExc_OverflowError);
        return s->e[0] != -1 || !PyErr_Occurred();
    }
    Ref f(PySequence_Fast(dims, "dims are an integer or a sequence of integers"));
    if (!f) return false;
    const Py_ssize_t n = PySequence_Fast_GET_SIZE(f.p);
    if (n > MOST) { PyErr_Format(PyExc_ValueError, "at most %lld dims are supported", g_max_dim); return false; }
    s->n = (int)n;
    for (Py_ssize_t i = 0; i < n; i++) {
        s->e[i] = PyNumber_AsSsize_t(PySequence_Fast_GET_ITEM(f.p, i), PyExc_OverflowError);
        if (s->e[i] == -1 && PyErr_Occurred()) return false;
    }
    return true;
}
bool var_shape(PyObject* v, Shape* s) {
    Ref a = attr(v, s_shape);
    return a && read_shape(a.p, s);
}
PyObject* shape_list(const Shape& s) {
    PyObject* l = PyList_New(s.n);
    if (!l) return nullptr;
    for (int i = 0; i < s.n; i++) {
        PyObject* v = PyLong_FromLongLong(s.e[i]);
        if (!v) { Py_DECREF(l); return nullptr; }
        PyList_SET_ITEM(l, i, v);
    }
    return l;
}
bool put(PyObject* d, PyObject* name, PyObject* stolen) {
    if (!stolen) return false;
    const int rc = PyDict_SetItem(d, name, stolen);
    Py_DECREF(stolen);
    return rc == 0;
}
PyObject* instance(PyTypeObject* t, PyObject** dict) {
    PyObject* o = t->tp_alloc(t, 0);
    if (!o) return nullptr;
    PyObject** dp = _PyObject_GetDictPtr(o);
    if (!*dp) *dp = _PyDict_NewPresized(8);
    if (!*dp) { Py_DECREF(o); return nullptr; }
    *dict = *dp;
    return o;
}

// ---- ops and Vars -----------------------------------------------------------------------------------------------------------
// Op.__init__: the inputs, who reads a Var (weakly: Var.assign moves them to the old value), the id, the register at creation
PyObject* new_op(PyTypeObject* type, PyObject* const* in, int n, PyObject** dict) {
    Ref op(instance(type, dict));
    if (!op) return nullptr;
    PyObject* list = PyList_New(n);
    if (!list) return nullptr;
    for (int i = 0; i < n; i++) PyList_SET_ITEM(list, i, keep(in[i]));
    if (!put(*dict, s_inputs, list)) return nullptr;
    Ref me(PyWeakref_NewRef(op.p, nullptr));
    if (!me) return nullptr;
    for (int i = 0; i < n; i++) {
        PyObject* lst = own(in[i], s__consumers);
        if (!lst || lst == Py_None) {
            PyObject* fresh = PyList_New(1);
            if (!fresh) return nullptr;
            PyList_SET_ITEM(fresh, 0, keep(me.p));
            if (!put(dict_of(in[i]), s__consumers, fresh)) return nullptr;
        } else {
            if (PyList_Append(lst, me.p)) return nullptr;
            const Py_ssize_t k = PyList_GET_SIZE(lst);
            if (k > 64 && (k & (k - 1)) == 0) {                // a long-lived var (a weight): drop the dead readers now and then
                Ref held(keep(lst)), alive(PyList_New(0));
                if (!alive) return nullptr;
                for (Py_ssize_t q = 0; q < PyList_GET_SIZE(lst); q++) {
                    PyObject* r = PyList_GET_ITEM(lst, q);
                    if (PyWeakref_GetObject(r) != Py_None && PyList_Append(alive.p, r)) return nullptr;
                }
                if (PyList_SetSlice(lst, 0, PyList_GET_SIZE(lst), alive.p)) return nullptr;
            }
        }
    }
    long long amp;
    if (amp_now(&amp)) return nullptr;
    if (!put(*dict, s_id, PyLong_FromLongLong(g_next_id++)) || !put(*dict, s_amp, PyLong_FromLongLong(amp & 63))) return nullptr;
    return op.give();
}
// Var(shape, dtype, op, num): the list is taken over
PyObject* new_var(PyObject* shape, PyObject* dtype, PyObject* op, long long num, bool scalar) {
    Ref sh(shape);
    if (!sh) return nullptr;
    PyObject* d;
    Ref v(instance(t_var, &d));
    if (!v) return nullptr;
    PyObject* od = dict_of(op);
    if (PyDict_SetItem(d, s_shape, sh.p) || !put(d, s_num, PyLong_FromLongLong(num)) || PyDict_SetItem(d, s_dtype, dtype) || PyDict_SetItem(d, s__op, op) ||
        !put(od, s__out_ref, PyWeakref_NewRef(v.p, nullptr)))
        return nullptr;
    PyObject* on = PyList_GET_ITEM(g_grad_enabled, 0);
    if (on == Py_True || (on != Py_False && PyObject_IsTrue(on) == 1)) {
        Ref ins(PyList_AsTuple(PyDict_GetItem(od, s_inputs)));
        if (!ins || !put(d, s__history, PyTuple_Pack(2, op, ins.p))) return nullptr;
    } else if (PyDict_SetItem(d, s__history, Py_None))
        return nullptr;
    if (!put(d, s_id, PyLong_FromLongLong(g_next_id++))) return nullptr;
    if (scalar && PyDict_SetItem(d, s_is_scalar, Py_True)) return nullptr;
    PyObject* co = PyDict_GetItemWithError(g_flags, s_compile_options);   // the flag's value at creation (var.cc:75)
    if (co && PyObject_IsTrue(co) == 1 && !put(d, s__compile_options, PyObject_CallOneArg((PyObject*)&PyDict_Type, co))) return nullptr;
    return v.give();
}
long long var_num(PyObject* v) {
    Ref n = attr(v, s_num);
    return n ? PyLong_AsLongLong(n.p) : -1;
}
PyObject* copy_shape(PyObject* v) {
    Ref a = attr(v, s_shape);
    return a ? PySequence_List(a.p) : nullptr;
}

// ---- numbers as Vars ----------------------------------------------------------------------------------------------------------
// the host Var of a Python number is kept by (type, value, sign[, dtype]): `x * 2.0` builds no new array each time
PyObject* number_var(PyObject* value, PyObject* dtype) {
    Ref sign(dtype || PyFloat_CheckExact(value) ? PyFloat_FromDouble(std::copysign(1.0, PyFloat_AsDouble(value))) : PyLong_FromLong(0));
    if (!sign || PyErr_Occurred()) return nullptr;
    Ref key(dtype ? PyTuple_Pack(4, (PyObject*)Py_TYPE(value), value, sign.p, dtype) : PyTuple_Pack(3, (PyObject*)Py_TYPE(value), value, sign.p));
    if (!key) return nullptr;
    if (PyObject* got = PyDict_GetItemWithError(g_scalars, key.p)) return keep(got);
    if (PyErr_Occurred()) return nullptr;
    if (PyDict_GET_SIZE(g_scalars) >= 4096) PyDict_Clear(g_scalars);
    Ref made(dtype ? PyObject_CallFunctionObjArgs(g_array, value, dtype, nullptr) : PyObject_CallOneArg(g_array, value));
    if (!made || PyDict_SetItem(g_scalars, key.p, made.p)) return nullptr;
    return made.give();
}
PyObject* as_var(PyObject* v) {
    if (is_var(v)) return keep(v);
    if (PyFloat_CheckExact(v) || PyLong_CheckExact(v) || PyBool_Check(v)) return number_var(v, nullptr);
    return PyObject_CallOneArg(g_as_var, v);
}

// ---- type rules -----------------------------------------------------------------------------------------------------------------
PyObject* binary_dtype(PyObject* op, PyObject* x, PyObject* y, bool xs, bool ys) {
    PyObject* dt = PyModule_GetDict(g_dt);
    PyObject *kept = PyDict_GetItem(dt, s__binary_dtypes), *amp = PyDict_GetItem(dt, s_amp_reg);
    PyObject *bx = xs ? Py_True : Py_False, *by = ys ? Py_True : Py_False;
    if (kept && amp) {
        Ref key(PyTuple_Pack(6, op, x, y, bx, by, amp));
        if (!key) return nullptr;
        if (PyObject* got = PyDict_GetItemWithError(kept, key.p)) return keep(got);
        if (PyErr_Occurred()) return nullptr;
    }
    Ref f(PyObject_GetAttr(g_dt, s_binary_dtype_infer));
    return f ? PyObject_CallFunctionObjArgs(f.p, op, x, y, bx, by, nullptr) : nullptr;
}
std::unordered_map<std::string, PyObject*> g_rules;          // unary and reduce rules by op, type and register (a few hundred at most)
PyObject* typed_rule(char kind, PyObject* op, PyObject* x, PyObject* function) {
    long long amp;
    Py_ssize_t n, m;
    const char *a = PyUnicode_AsUTF8AndSize(op, &n), *b = a ? PyUnicode_AsUTF8AndSize(x, &m) : nullptr;
    if (!b || amp_now(&amp)) return nullptr;
    std::string key(1, kind);
    key.append(a, n).append(1, '\0').append(b, m).append(1, '\0').append((const char*)&amp, sizeof amp);
    auto it = g_rules.find(key);
    if (it != g_rules.end()) return keep(it->second);
    Ref f(PyObject_GetAttr(g_dt, function));
    Ref got(f ? PyObject_CallFunctionObjArgs(f.p, op, x, nullptr) : nullptr);
    long long after;
    if (!got || amp_now(&after)) return nullptr;
    if (after == amp && g_rules.size() < 4096) g_rules.emplace(std::move(key), keep(got.p));    // (another thread may have set the register meanwhile)
    return got.give();
}

// ---- constructors ---------------------------------------------------------------------------------------------------------------
PyObject* make_cast(PyObject* x, PyObject* op, PyObject* dtype) {
    PyObject* d;
    Ref o(new_op(t_unary, &x, 1, &d));
    if (!o || PyDict_SetItem(d, s_op, op)) return nullptr;
    const long long num = var_num(x);
    if (num < 0) return nullptr;
    return new_var(copy_shape(x), dtype, o.p, num, flag(x, s_is_scalar));
}
PyObject* unary(PyObject* x0, PyObject* op, PyObject* force, bool forward) {
    Ref x(as_var(x0));
    if (!x) return nullptr;
    int is = PySet_Contains(g_dtypes, op);
    if (is < 0) return nullptr;
    if (is && PyUnicode_Compare(op, s_void) != 0) {
        Ref have = attr(x.p, s_dtype);
        if (!have) return nullptr;
        if (forward && PyUnicode_Compare(op, have.p) == 0) return x.give();                    // forward(x), unary_op.cc:867-870
        return make_cast(x.p, s_cast, op);
    }
    if (force != Py_None && PyUnicode_Check(op) && PyUnicode_Compare(op, s_cast) == 0) return make_cast(x.p, op, force);
    is = PySet_Contains(g_unary_ops, op);
    if (is < 0) return nullptr;
    if (!is) return PyErr_Format(PyExc_ValueError, "unknown unary op %R", op);
    Ref have = attr(x.p, s_dtype);
    Ref dtype(have ? typed_rule('u', op, have.p, s_unary_dtype_infer) : nullptr);
    return dtype ? make_cast(x.p, op, dtype.p) : nullptr;
}

// infer_shape of ops/broadcast_to_op.cc:119-168: the result's extents, the masks with the implicit broadcasts added
bool broadcast_rule(const Shape& x, const Shape& y, long long* bmask, long long* kmask, Shape* z, long long* num) {
    const int cnt = __builtin_popcountll((unsigned long long)(*bmask & ~*kmask));
    const int zdim = std::max(x.n, y.n - cnt) + cnt;
    if (zdim > MOST) { PyErr_Format(PyExc_ValueError, "at most %lld dims are supported", g_max_dim); return false; }
    z->n = zdim;
    int xi = x.n - 1, yi = y.n - 1;
    for (int i = zdim - 1; i >= 0; i--) {
        const bool bx = xi >= 0, by = yi >= 0;
        const long long xs = bx ? x.e[xi] : 1, ys = by ? y.e[yi] : 1;
        if (*bmask >> i & 1) {
            yi--;
            if (*kmask >> i & 1) xi--;
            z->e[i] = ys;
            continue;
        }
        const long long m = (long long)(xs == 1 && (ys != 1 || !bx)) << i;
        *bmask |= m;
        if (bx) *kmask |= m;
        long long zs = xs;
        if ((xs == 1 || ys == 1) && xs != ys)
            zs = xs * ys;
        else if (xs != ys) {
            Ref a(shape_list(x)), b(shape_list(y));
            if (a && b) PyErr_Format(PyExc_ValueError, "Shape not match %R %R", a.p, b.p);
            return false;
        }
        z->e[i] = zs;
        xi--;
        yi--;
    }
    if (zdim > g_max_dim) { PyErr_Format(PyExc_ValueError, "at most %lld dims are supported", g_max_dim); return false; }
    for (int i = 0; i < zdim; i++)
        if (z->e[i] < 0) {
            Ref a(shape_list(*z));
            if (a) PyErr_Format(PyExc_ValueError, "Shape should greater than 0: %R", a.p);
            return false;
        }
    return count_elements(*z, num);
}
PyObject* broadcast_to(PyObject* x, const Shape& xs, const Shape& shape, long long bmask, long long kmask) {
    Shape z;
    long long num;
    if (!broadcast_rule(xs, shape, &bmask, &kmask, &z, &num)) return nullptr;
    PyObject* d;
    Ref o(new_op(t_broadcast, &x, 1, &d));
    if (!o || !put(d, s_bcast_mask, PyLong_FromLongLong(bmask)) || !put(d, s_keepdims_mask, PyLong_FromLongLong(kmask))) return nullptr;
    Ref dtype = attr(x, s_dtype);
    return dtype ? new_var(shape_list(z), dtype.p, o.p, num, flag(x, s_is_scalar)) : nullptr;
}
// ops/broadcast_to_op.cc:98-103
bool need_broadcast(const Shape& x, const Shape& y) {
    if (x.n < y.n) return true;
    for (int i = 1; i <= y.n; i++)
        if (x.e[x.n - i] != y.e[y.n - i] && y.e[y.n - i] != 1) return true;
    return false;
}
// broadcast without named axes
PyObject* broadcast_plain(PyObject* x, const Shape& shape) {
    Shape xs;
    if (!var_shape(x, &xs)) return nullptr;
    if (!need_broadcast(xs, shape)) return keep(x);            // forward(x)
    if (shape.n == 0) return PyErr_Format(PyExc_ValueError, "Number of shape should greater than 0.");
    for (int i = 0; i < shape.n; i++)
        if (shape.e[i] < 0) return PyErr_Format(PyExc_ValueError, "Shape should greater than 0.");
    return broadcast_to(x, xs, shape, 0, 0);
}
PyObject* same_shape_binary(PyObject* x, PyObject* y, PyObject* op) {
    Ref dx = attr(x, s_dtype), dy = attr(y, s_dtype);
    if (!dx || !dy) return nullptr;
    Ref dtype(binary_dtype(op, dx.p, dy.p, flag(x, s_is_scalar), flag(y, s_is_scalar)));
    if (!dtype) return nullptr;
    PyObject* in[2] = {x, y};
    PyObject* d;
    Ref o(new_op(t_binary, in, 2, &d));
    if (!o || PyDict_SetItem(d, s_op, op)) return nullptr;
    const long long num = var_num(x);
    return num < 0 ? nullptr : new_var(copy_shape(x), dtype.p, o.p, num, false);
}
PyObject* binary(PyObject* x0, PyObject* y0, PyObject* op) {
    Ref x(as_var(x0));
    if (!x) return nullptr;
    Ref y(as_var(y0));
    if (!y) return nullptr;
    const int is = PySet_Contains(g_binary_ops, op);
    if (is < 0) return nullptr;
    if (!is) return PyErr_Format(PyExc_ValueError, "unknown binary op %R", op);
    Shape xs, ys;
    if (!var_shape(x.p, &xs) || !var_shape(y.p, &ys)) return nullptr;
    if (xs == ys) return same_shape_binary(x.p, y.p, op);
    // broadcasts are inserted when ranks differ or an extent is 1 on one side only; other mismatches are errors
    for (int i = 1; i <= std::min(xs.n, ys.n); i++) {
        const long long a = xs.e[xs.n - i], b = ys.e[ys.n - i];
        if (a != b && a != 1 && b != 1) {
            Ref p(shape_list(xs)), q(shape_list(ys));
            return p && q ? PyErr_Format(PyExc_ValueError, "Shape not match, x:%R y:%R", p.p, q.p) : nullptr;
        }
    }
    Ref xp(broadcast_plain(x.p, ys));
    if (!xp) return nullptr;
    Ref yp(broadcast_plain(y.p, xs));
    if (!yp) return nullptr;
    if (Py_EnterRecursiveCall(" while shapes are matched")) return nullptr;
    PyObject* z = binary(xp.p, yp.p, op);
    Py_LeaveRecursiveCall();
    return z;
}
PyObject* ternary(PyObject* c0, PyObject* x0, PyObject* y0) {
    Ref v[3] = {Ref(as_var(c0)), Ref(), Ref()};
    if (!v[0]) return nullptr;
    v[1] = Ref(as_var(x0));
    if (!v[1]) return nullptr;
    v[2] = Ref(as_var(y0));
    if (!v[2]) return nullptr;
    Shape s[3];
    for (int i = 0; i < 3; i++)
        if (!var_shape(v[i].p, &s[i])) return nullptr;
    if (!(s[0] == s[1] && s[0] == s[2])) {
        auto num = [&](int i) { return var_num(v[i].p); };
        auto larger = [&](int a, int b) { return s[a].n > s[b].n || num(a) > num(b); };
        if (larger(0, 1) || larger(0, 2) || larger(1, 0) || larger(2, 0)) {
            auto spread = [&](int which, int to) {
                Ref z(broadcast_plain(v[which].p, s[to]));
                if (!z || !var_shape(z.p, &s[which])) return false;
                v[which] = std::move(z);
                return true;
            };
            const bool bx2 = larger(1, 0), by2 = larger(2, 0);
            if (bx2 && !spread(0, 1)) return nullptr;
            if (by2 && !spread(0, 2)) return nullptr;
            const bool bx = larger(0, 1), by = larger(0, 2);
            if (bx && !spread(1, 0)) return nullptr;
            if (by && !spread(2, 0)) return nullptr;
            if (Py_EnterRecursiveCall(" while shapes are matched")) return nullptr;      // (no extents and one do not meet)
            PyObject* z = ternary(v[0].p, v[1].p, v[2].p);
            Py_LeaveRecursiveCall();
            return z;
        }
        if (!(s[0].n == s[1].n && s[0].n == s[2].n)) return PyErr_Format(PyExc_ValueError, "Number of dims should be the same.");
        Ref a(shape_list(s[1])), b(shape_list(s[2])), c(shape_list(s[0]));
        return a && b && c ? PyErr_Format(PyExc_ValueError, "Shape not match %R %R %R", a.p, b.p, c.p) : nullptr;
    }
    Ref dx = attr(v[1].p, s_dtype), dy = attr(v[2].p, s_dtype);
    if (!dx || !dy) return nullptr;
    Ref dtype;
    if (PyUnicode_Compare(dx.p, dy.p) == 0)
        dtype = Ref(keep(dx.p));
    else {
        Ref f(PyObject_GetAttr(g_dt, s_dtype_infer));
        dtype = Ref(f ? PyObject_CallFunctionObjArgs(f.p, dx.p, dy.p, flag(v[1].p, s_is_scalar) ? Py_True : Py_False, flag(v[2].p, s_is_scalar) ? Py_True : Py_False, nullptr) : nullptr);
    }
    if (!dtype) return nullptr;
    PyObject* in[3] = {v[0].p, v[1].p, v[2].p};
    PyObject* d;
    Ref o(new_op(t_ternary, in, 3, &d));
    if (!o) return nullptr;
    const long long num = var_num(v[1].p);
    return num < 0 ? nullptr : new_var(copy_shape(v[1].p), dtype.p, o.p, num, false);
}
PyObject* reduce_mask(PyObject* x, PyObject* op, long long rmask, long long kmask) {
    long long amp;
    if (amp_now(&amp)) return nullptr;
    Ref have = attr(x, s_dtype);
    if (!have) return nullptr;
    auto is = [](PyObject* a, PyObject* b) { return PyUnicode_Compare(a, b) == 0; };
    if (!(amp & 32) && (is(have.p, s_float16) || is(have.p, s_bfloat16)) && (is(op, s_mean) || is(op, s_add))) {
        // improve 16-bit float precision: cast -> reduce -> cast (reduce_op.cc:259-266, 295-302)
        Ref wide(unary(x, s_float32, Py_None, true));
        Ref sum(wide ? reduce_mask(wide.p, op, rmask, kmask) : nullptr);
        return sum ? unary(sum.p, have.p, Py_None, true) : nullptr;
    }
    Shape xs, z;
    if (!var_shape(x, &xs)) return nullptr;
    long long num;
    for (int i = 0; i < xs.n; i++) {
        if (rmask >> i & 1) {
            if (kmask >> i & 1) z.e[z.n++] = 1;
        } else
            z.e[z.n++] = xs.e[i];
    }
    if (!z.n) {
        z.e[z.n++] = 1;
        kmask |= 1;
    }
    if (!count_elements(z, &num)) return nullptr;
    Ref dtype(typed_rule('r', op, have.p, s_reduce_dtype_infer));
    if (!dtype) return nullptr;
    PyObject* d;
    Ref o(new_op(t_reduce, &x, 1, &d));
    if (!o || PyDict_SetItem(d, s_op, op) || !put(d, s_reduce_mask, PyLong_FromLongLong(rmask)) || !put(d, s_keepdims_mask, PyLong_FromLongLong(kmask))) return nullptr;
    return new_var(shape_list(z), dtype.p, o.p, num, z.n == 1 && num == 1);
}

// ---- argument lists ---------------------------------------------------------------------------------------------------------------
// positional and keyword arguments into out[0..n) (borrowed; what is not given stays as it is)
bool arguments(const char* name, PyObject* const* args, Py_ssize_t nargs, PyObject* kw, const char* const* names, int n, int least, PyObject** out) {
    if (nargs > n) { PyErr_Format(PyExc_TypeError, "%s() takes at most %d arguments (%zd given)", name, n, nargs); return false; }
    for (Py_ssize_t i = 0; i < nargs; i++) out[i] = args[i];
    bool given[8] = {};
    for (Py_ssize_t i = 0; i < nargs; i++) given[i] = true;
    if (kw)
        for (Py_ssize_t k = 0; k < PyTuple_GET_SIZE(kw); k++) {
            int at = -1;
            for (int i = 0; i < n; i++)
                if (PyUnicode_CompareWithASCIIString(PyTuple_GET_ITEM(kw, k), names[i]) == 0) at = i;
            if (at < 0 || given[at]) { PyErr_Format(PyExc_TypeError, "%s() got an unexpected or repeated argument %R", name, PyTuple_GET_ITEM(kw, k)); return false; }
            given[at] = true;
            out[at] = args[nargs + k];
        }
    for (int i = 0; i < least; i++)
        if (!given[i]) { PyErr_Format(PyExc_TypeError, "%s() missing argument '%s'", name, names[i]); return false; }
    return true;
}
#define FUNCTION(name) PyObject* py_##name(PyObject*, PyObject* const* args, Py_ssize_t nargs, PyObject* kw)

FUNCTION(unary) {
    static const char* const names[] = {"x", "op", "force_dtype", "allow_forward"};
    PyObject* a[4] = {nullptr, nullptr, Py_None, Py_True};
    if (!arguments("unary", args, nargs, kw, names, 4, 2, a)) return nullptr;
    return unary(a[0], a[1], a[2], PyObject_IsTrue(a[3]) == 1);
}
FUNCTION(binary) {
    static const char* const names[] = {"x", "y", "op"};
    PyObject* a[3];
    return arguments("binary", args, nargs, kw, names, 3, 3, a) ? binary(a[0], a[1], a[2]) : nullptr;
}
FUNCTION(ternary) {
    static const char* const names[] = {"cond", "x", "y"};
    PyObject* a[3];
    return arguments("ternary", args, nargs, kw, names, 3, 3, a) ? ternary(a[0], a[1], a[2]) : nullptr;
}
FUNCTION(broadcast) {
    static const char* const names[] = {"x", "shape", "dims"};
    PyObject* a[3] = {nullptr, nullptr, nullptr};
    if (!arguments("broadcast", args, nargs, kw, names, 3, 2, a)) return nullptr;
    Ref x(as_var(a[0]));
    if (!x) return nullptr;
    Shape shape, xs, dims;
    if (is_var(a[1]) ? !var_shape(a[1], &shape) : !read_shape(a[1], &shape)) return nullptr;
    if (a[2] && !read_dims(a[2], &dims)) return nullptr;
    if (!dims.n) return broadcast_plain(x.p, shape);
    if (!var_shape(x.p, &xs)) return nullptr;
    if (shape.n == 0) return PyErr_Format(PyExc_ValueError, "Number of shape should greater than 0.");
    for (int i = 0; i < shape.n; i++)
        if (shape.e[i] < 0) return PyErr_Format(PyExc_ValueError, "Shape should greater than 0.");
    const int ydim = std::max(xs.n, shape.n - dims.n) + dims.n;
    long long bmask = 0;
    for (int i = 0; i < dims.n; i++) {
        const long long d = dims.e[i] < 0 ? dims.e[i] + ydim : dims.e[i];
        if (d < 0 || d >= ydim || d > 62) {
            Ref l(shape_list(dims));
            return l ? PyErr_Format(PyExc_ValueError, "Wrong dims number: %R", l.p) : nullptr;
        }
        bmask |= 1ll << d;
    }
    return broadcast_to(x.p, xs, shape, bmask, 0);
}
// make_broadcast_to(x, shape, dims_mask, keepdims_mask), used by gradients
FUNCTION(broadcast_mask) {
    static const char* const names[] = {"x", "shape", "bmask", "kmask"};
    PyObject* a[4];
    if (!arguments("_broadcast_mask", args, nargs, kw, names, 4, 4, a)) return nullptr;
    const long long bmask = PyLong_AsLongLong(a[2]), kmask = PyLong_AsLongLong(a[3]);
    if (PyErr_Occurred()) return nullptr;
    if (!bmask) return keep(a[0]);
    Shape xs, shape;
    if (!var_shape(a[0], &xs) || !read_shape(a[1], &shape)) return nullptr;
    return broadcast_to(a[0], xs, shape, bmask, kmask);
}
FUNCTION(reduce) {
    static const char* const names[] = {"x", "op", "dims", "keepdims"};
    PyObject* a[4] = {nullptr, nullptr, nullptr, Py_False};
    if (!arguments("reduce", args, nargs, kw, names, 4, 2, a)) return nullptr;
    Ref x(as_var(a[0]));
    if (!x) return nullptr;
    int is = PySet_Contains(g_binary_ops, a[1]);
    if (is < 0) return nullptr;
    if (!is) return PyErr_Format(PyExc_ValueError, "unknown reduce op %R", a[1]);
    is = PySet_Contains(g_reduce_ops, a[1]);
    if (is < 0) return nullptr;
    if (!is) return PyErr_Format(PyExc_ValueError, "reduce op %R is not associative; not supported on the device", a[1]);
    Shape xs, dims;
    if (!var_shape(x.p, &xs)) return nullptr;
    if (a[2] && !read_dims(a[2], &dims)) return nullptr;
    long long rmask = dims.n ? 0 : (1ll << xs.n) - 1;
    for (int i = 0; i < dims.n; i++) {
        const long long d = dims.e[i] < 0 ? dims.e[i] + xs.n : dims.e[i];
        if (d < 0 || d >= xs.n) {
            Ref l(shape_list(dims));
            return l ? PyErr_Format(PyExc_ValueError, "Wrong dims number: %R", l.p) : nullptr;
        }
        rmask |= 1ll << d;
    }
    const int keepdims = PyObject_IsTrue(a[3]);
    return keepdims < 0 ? nullptr : reduce_mask(x.p, a[1], rmask, keepdims ? (1ll << 30) - 1 : 0);
}
FUNCTION(reduce_mask) {
    static const char* const names[] = {"x", "op", "rmask", "kmask"};
    PyObject* a[4];
    if (!arguments("_reduce_mask", args, nargs, kw, names, 4, 4, a)) return nullptr;
    const long long rmask = PyLong_AsLongLong(a[2]), kmask = PyLong_AsLongLong(a[3]);
    return PyErr_Occurred() ? nullptr : reduce_mask(a[0], a[1], rmask, kmask);
}
// ops/op_utils.cc:19-36: a [1] array of like's dtype broadcast to like
FUNCTION(make_number) {
    static const char* const names[] = {"value", "like"};
    PyObject* a[2];
    if (!arguments("make_number", args, nargs, kw, names, 2, 2, a)) return nullptr;
    Shape s;
    Ref dtype = attr(a[1], s_dtype);
    if (!dtype || !var_shape(a[1], &s)) return nullptr;
    if (s.n == 1 && s.e[0] == 1) return PyObject_CallFunctionObjArgs(g_array, a[0], dtype.p, nullptr);     // nothing to spread: the caller's own Var
    Ref v(PyFloat_CheckExact(a[0]) || PyLong_CheckExact(a[0]) ? number_var(a[0], dtype.p) : PyObject_CallFunctionObjArgs(g_array, a[0], dtype.p, nullptr));
    return v ? broadcast_plain(v.p, s) : nullptr;
}
PyObject* py_new_id(PyObject*, PyObject*) { return PyLong_FromLongLong(g_next_id++); }

// ---- gradients ------------------------------------------------------------------------------------------------------------------
bool is_float_name(PyObject* dtype) {
    const char* p = PyUnicode_AsUTF8(dtype);
    return p && (!strncmp(p, "float", 5) || !strcmp(p, "bfloat16"));
}
long long id_of(PyObject* v) {
    PyObject* i = own(v, s_id);
    return i ? PyLong_AsLongLong(i) : -1;
}
bool in_set(PyObject* set, PyObject* v) {
    PyObject* i = own(v, s_id);
    return i && PySet_Contains(set, i) == 1;
}
bool is_text(PyObject* s, const char* t) { return s && PyUnicode_Check(s) && PyUnicode_CompareWithASCIIString(s, t) == 0; }
PyObject* number_like(double value, bool whole, PyObject* like) {
    Shape s;
    Ref dtype = attr(like, s_dtype);
    if (!dtype || !var_shape(like, &s)) return nullptr;
    Ref n(whole ? PyLong_FromLong((long)value) : PyFloat_FromDouble(value));
    if (!n) return nullptr;
    if (s.n == 1 && s.e[0] == 1) return PyObject_CallFunctionObjArgs(g_array, n.p, dtype.p, nullptr);
    Ref v(number_var(n.p, dtype.p));
    return v ? broadcast_plain(v.p, s) : nullptr;
}
PyObject *s_multiply, *s_divide, *s_subtract, *s_negative, *s_equal;
// factor * dout, which is `factor` itself where dout is the seed of this call, spread or cast: the product would be a pass over memory that
// changes nothing (the gradient of a 32 x 128 x 56 x 56 float32 result under (y * g).sum(): 19 us).  `ones` holds the ids of those Vars; a Var of the program's own that happens to hold a 1 is not among them, whatever its
// value, since a second derivative may ask for it.  A factor that is spread or gathered stays a product: it is how the operands of
// convolutions and matrix products appear, which are recognised by it.
PyObject* times(PyObject* factor, PyObject* dout, PyObject* ones) {
    if (in_set(ones, dout)) {
        PyObject* op = own(factor, s__op);
        if (!op || !(PyObject_TypeCheck(op, t_broadcast) || PyObject_TypeCheck(op, t_reindex))) {
            Ref a = attr(factor, s_dtype), b = attr(dout, s_dtype);
            Ref z(a && b ? binary_dtype(s_multiply, a.p, b.p, flag(factor, s_is_scalar), flag(dout, s_is_scalar)) : nullptr);
            if (!z) return nullptr;
            if (PyUnicode_Compare(z.p, a.p) == 0) return keep(factor);
        }
    }
    return binary(factor, dout, s_multiply);
}
// the gradient of input `index` of an op with result `out` (new reference; None: no gradient).  What is not here is grad.py's.
PyObject* op_gradient(PyObject* op, PyObject* inputs, PyObject* out, PyObject* dout, Py_ssize_t index, PyObject* ones, PyObject* others) {
    PyTypeObject* t = Py_TYPE(op);
    PyObject* x = PyTuple_GET_ITEM(inputs, 0);
    PyObject* name = own(op, s_op);
    auto still_one = [&](PyObject* v) {                        // v is dout, spread or cast
        if (v && in_set(ones, dout)) {
            PyObject* i = own(v, s_id);
            if (PySet_Add(ones, i)) { Py_DECREF(v); return (PyObject*)nullptr; }
        }
        return v;
    };
    if (t == t_unary) {
        Ref dtype = attr(x, s_dtype);
        if (!dtype) return nullptr;
        if (!is_float_name(dtype.p)) Py_RETURN_NONE;
        if (is_text(name, "cast")) return still_one(unary(dout, dtype.p, Py_None, true));
        if (is_text(name, "negative")) return unary(dout, s_negative, Py_None, true);
        if (is_text(name, "exp")) return binary(dout, out, s_multiply);
        if (is_text(name, "log")) return binary(dout, x, s_divide);
        if (is_text(name, "sqrt")) {
            Ref two(number_like(2, true, x));
            Ref d(two ? binary(two.p, out, s_multiply) : nullptr);
            return d ? binary(dout, d.p, s_divide) : nullptr;
        }
        if (is_text(name, "sigmoid")) {
            Ref sq(binary(out, out, s_multiply));
            Ref d(sq ? binary(out, sq.p, s_subtract) : nullptr);
            return d ? binary(dout, d.p, s_multiply) : nullptr;
        }
    } else if (t == t_binary) {
        PyObject* y = PyTuple_GET_ITEM(inputs, 1);
        if (is_text(name, "add")) return keep(dout);
        if (is_text(name, "subtract")) return index == 0 ? keep(dout) : unary(dout, s_negative, Py_None, true);
        if (is_text(name, "multiply")) return times(index == 0 ? y : x, dout, ones);
        if (is_text(name, "divide")) {
            if (index == 0) return binary(dout, y, s_divide);
            Ref n(unary(dout, s_negative, Py_None, true));
            Ref a(n ? binary(n.p, x, s_multiply) : nullptr);
            Ref b(a ? binary(y, y, s_multiply) : nullptr);
            return b ? binary(a.p, b.p, s_divide) : nullptr;
        }
    } else if (t == t_ternary) {                               // ops/ternary_op.cc:49-56
        if (index == 0) Py_RETURN_NONE;
        Ref zeros(number_like(0, true, dout));
        if (!zeros) return nullptr;
        return index == 1 ? ternary(x, dout, zeros.p) : ternary(x, zeros.p, dout);
    } else if (t == t_broadcast) {                             // ops/broadcast_to_op.cc:112-117
        const long long b = PyLong_AsLongLong(own(op, s_bcast_mask)), k = PyLong_AsLongLong(own(op, s_keepdims_mask));
        return b ? reduce_mask(dout, s_add, b, k) : keep(dout);
    } else if (t == t_reduce) {                                // ops/reduce_op.cc:339-362
        Shape xs;
        const long long b = PyLong_AsLongLong(own(op, s_reduce_mask)), k = PyLong_AsLongLong(own(op, s_keepdims_mask));
        if (!var_shape(x, &xs)) return nullptr;
        auto bc = [&](PyObject* v) -> PyObject* {
            Shape vs;
            if (!b) return keep(v);
            return var_shape(v, &vs) ? broadcast_to(v, vs, xs, b, k) : nullptr;
        };
        if (is_text(name, "add")) return still_one(bc(dout));
        if (is_text(name, "mean")) {
            Ref a(bc(dout));
            Ref n(a ? number_like(1.0 * (double)var_num(out) / (double)var_num(x), false, a.p) : nullptr);
            return n ? binary(a.p, n.p, s_multiply) : nullptr;
        }
        if (is_text(name, "maximum") || is_text(name, "minimum")) {
            Ref m(bc(out));
            Ref cond(m ? binary(x, m.p, s_equal) : nullptr);
            Ref d(cond ? bc(dout) : nullptr);
            Ref zero(d ? number_like(0, true, x) : nullptr);
            return zero ? ternary(cond.p, d.p, zero.p) : nullptr;
        }
    }
    Ref i(PyLong_FromSsize_t(index));
    return i ? PyObject_CallFunctionObjArgs(others, op, inputs, out, dout, i.p, nullptr) : nullptr;
}
typedef std::unordered_map<long long, Ref> Grads;
// The gradients of the Vars in `dep` by id.  `ones` takes the ids of the seed and of what is only it, spread or cast, so that products
// with it are left out; where `fold` is not set it stays empty.
bool backward(PyObject* loss, const std::vector<std::pair<long long, Ref>>& order, const std::unordered_set<long long>& dep, PyObject* ones, bool fold, PyObject* others, Grads* grads) {
    if (dep.count(id_of(loss))) {
        PyObject* seed = number_like(1.0, false, loss);
        if (!seed) return false;
        (*grads)[id_of(loss)] = Ref(seed);
        if (fold && PySet_Add(ones, own(seed, s_id))) return false;
    }
    PyObject* dt = PyModule_GetDict(g_dt);
    for (size_t q = order.size(); q-- > 0;) {
        PyObject* v = order[q].second.p;
        auto it = grads->find(order[q].first);
        PyObject* h = own(v, s__history);
        if (it == grads->end() || !h || h == Py_None) continue;
        Ref g(keep(it->second.p)), history(keep(h));
        PyObject *op = PyTuple_GET_ITEM(h, 0), *inputs = PyTuple_GET_ITEM(h, 1);
        for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(inputs); i++) {
            PyObject* u = PyTuple_GET_ITEM(inputs, i);
            const long long uid = id_of(u);
            if (!dep.count(uid)) continue;
            Ref type = attr(u, s_dtype);
            if (!type) return false;
            if (!is_float_name(type.p)) continue;
            // an op's gradient is built under the register the op was created with (grad.cc:48-55)
            long long saved;
            if (amp_now(&saved)) return false;
            PyObject* mine = own(op, s_amp);
            const long long amp = saved | (mine ? PyLong_AsLongLong(mine) : 0);
            Ref before(keep(PyDict_GetItem(dt, s_amp_reg)));
            if (amp != saved && !put(dt, s_amp_reg, PyLong_FromLongLong(amp))) return false;
            Ref du(op_gradient(op, inputs, v, g.p, i, ones, others));
            if (amp != saved) {
                PyObject *et, *ev, *tb;
                PyErr_Fetch(&et, &ev, &tb);
                if (PyDict_SetItem(dt, s_amp_reg, before.p)) return false;
                PyErr_Restore(et, ev, tb);
            }
            if (!du) return false;
            if (du.p == Py_None) continue;
            Shape ds, us;
            if (!var_shape(du.p, &ds) || !var_shape(u, &us)) return false;
            if (!(ds == us)) {
                Ref a(shape_list(ds)), b(shape_list(us));
                if (a && b) PyErr_Format(PyExc_RuntimeError, "gradient of %R has shape %R, expected %R", op, a.p, b.p);
                return false;
            }
            auto at = grads->find(uid);
            if (at == grads->end()) grads->emplace(uid, std::move(du));
            else {
                PyObject* sum = binary(at->second.p, du.p, s_add);
                if (!sum) return false;
                grads->find(uid)->second = Ref(sum);
            }
        }
    }
    return true;
}
// gradients(loss, targets, others): a list, one Var per target (grad.cc:85-284); others(op, inputs, out, dout, index) for ops not covered here.
PyObject* py_gradients(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    if (nargs != 3 || !is_var(args[0]) || !PyList_Check(args[1])) return PyErr_Format(PyExc_TypeError, "gradients(loss, targets, others)");
    PyObject *loss = args[0], *targets = args[1];
    // vars the loss depends on, through retained history
    std::unordered_set<long long> nodes, dep, wanted;
    std::vector<std::pair<long long, Ref>> order;
    std::vector<PyObject*> stack{loss};                        // (held by the histories of the vars in `order`)
    while (!stack.empty()) {
        PyObject* v = stack.back();
        stack.pop_back();
        const long long id = id_of(v);
        if (!nodes.insert(id).second) continue;
        order.emplace_back(id, Ref(keep(v)));
        PyObject* h = own(v, s__history);
        if (!h || h == Py_None) continue;
        PyObject* inputs = PyTuple_GET_ITEM(h, 1);
        for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(inputs); i++)
            if (!nodes.count(id_of(PyTuple_GET_ITEM(inputs, i)))) stack.push_back(PyTuple_GET_ITEM(inputs, i));
    }
    // of those, the ones that depend on a target (ids grow from inputs to outputs)
    std::sort(order.begin(), order.end(), [](const auto& a, const auto& b) { return a.first < b.first; });
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(targets); i++) wanted.insert(id_of(PyList_GET_ITEM(targets, i)));
    for (auto& [id, v] : order) {
        if (wanted.count(id)) {
            dep.insert(id);
            continue;
        }
        PyObject* h = own(v.p, s__history);
        if (!h || h == Py_None) continue;
        PyObject* inputs = PyTuple_GET_ITEM(h, 1);
        for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(inputs); i++)
            if (dep.count(id_of(PyTuple_GET_ITEM(inputs, i)))) {
                dep.insert(id);
                break;
            }
    }
    Grads grads;
    Ref ones(PySet_New(nullptr));
    if (!ones || !backward(loss, order, dep, ones.p, true, args[2], &grads)) return nullptr;
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(targets); i++) {
        auto it = grads.find(id_of(PyList_GET_ITEM(targets, i)));
        if (it != grads.end() && in_set(ones.p, it->second.p)) {
            // the caller gets hold of the seed (or of it spread or cast) and may ask for derivatives by it: nothing is left out then
            grads.clear();
            ones = Ref(PyFrozenSet_New(nullptr));
            if (!ones || !backward(loss, order, dep, ones.p, false, args[2], &grads)) return nullptr;
            break;
        }
    }
    Ref out(PyList_New(0));
    if (!out) return nullptr;
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(targets); i++) {
        PyObject* t = PyList_GET_ITEM(targets, i);
        auto it = grads.find(id_of(t));
        Ref g;
        if (it == grads.end()) g = Ref(number_like(0.0, false, t));
        else if (nodes.count(id_of(it->second.p))) {           // a var of the caller's own: the gradient is a var of its own
            Ref dtype = attr(it->second.p, s_dtype);
            g = Ref(dtype ? unary(it->second.p, s_cast, dtype.p, false) : nullptr);
        } else
            g = Ref(keep(it->second.p));
        if (!g || PyList_Append(out.p, g.p)) return nullptr;
    }
    return out.give();
}

// ---- pending ops ----------------------------------------------------------------------------------------------------------------
// Pending producers behind `targets`, in topological order.
PyObject* py_pending_ops(PyObject*, PyObject* targets) {
    Ref f(PySequence_Fast(targets, "targets"));
    Ref order(PyList_New(0));
    if (!f || !order) return nullptr;
    // (every op on the stack is held by its result, which is a target or the input of an op further down)
    std::vector<std::pair<PyObject*, bool>> stack;             // op, its inputs have been visited
    std::unordered_set<PyObject*> seen;
    for (Py_ssize_t i = 0; i < PySequence_Fast_GET_SIZE(f.p); i++) {
        PyObject* v = PySequence_Fast_GET_ITEM(f.p, i);
        PyObject* op = own(v, s__op);
        if (absent(v, s__buf) && op && op != Py_None) stack.push_back({op, false});
    }
    while (!stack.empty()) {
        auto [op, visited] = stack.back();
        if (visited) {
            stack.pop_back();
            if (seen.insert(op).second && PyList_Append(order.p, op)) return nullptr;
            continue;
        }
        if (seen.count(op)) {
            stack.pop_back();
            continue;
        }
        stack.back().second = true;
        PyObject* ins = own(op, s_inputs);
        if (!ins || !PyList_Check(ins)) { PyErr_SetString(PyExc_TypeError, "an op's inputs are a list"); return nullptr; }
        for (Py_ssize_t i = 0; i < PyList_GET_SIZE(ins); i++) {
            PyObject* u = PyList_GET_ITEM(ins, i);
            if (!absent(u, s__buf)) continue;
            PyObject* p = own(u, s__op);
            if (p && p != Py_None && !seen.count(p)) stack.push_back({p, false});
        }
    }
    return order.give();
}

// ---- the key of a graph ---------------------------------------------------------------------------------------------------------
struct Key {
    std::string b;
    void num(long long v) {                                    // 7 bits at a time, the sign folded in
        unsigned long long u = ((unsigned long long)v << 1) ^ (unsigned long long)(v >> 63);
        while (u >= 0x80) {
            b.push_back((char)(u | 0x80));
            u >>= 7;
        }
        b.push_back((char)u);
    }
    bool text(PyObject* s) {
        Py_ssize_t n;
        if (!s) { PyErr_SetString(PyExc_AttributeError, "an op without what it was made with"); return false; }
        const char* p = PyUnicode_AsUTF8AndSize(s, &n);
        if (!p) return false;
        num(n);
        b.append(p, (size_t)n);
        return true;
    }
    bool texts(PyObject* l) {
        if (!l) return text(l);
        Ref f(PySequence_Fast(l, "a list of expressions"));
        if (!f) return false;
        num(PySequence_Fast_GET_SIZE(f.p));
        for (Py_ssize_t i = 0; i < PySequence_Fast_GET_SIZE(f.p); i++)
            if (!text(PySequence_Fast_GET_ITEM(f.p, i))) return false;
        return true;
    }
    bool integer(PyObject* v) {
        if (!v) return text(v);
        const long long n = PyLong_AsLongLong(v);
        if (n == -1 && PyErr_Occurred()) return false;
        num(n);
        return true;
    }
    bool var(PyObject* v) {                                    // shape and type
        Shape s;
        Ref t = attr(v, s_dtype);
        if (!t || !var_shape(v, &s)) return false;
        num(s.n);
        for (int i = 0; i < s.n; i++) num(s.e[i]);
        return text(t.p);
    }
};
// A one-element host array whose bytes are all zero.  Values are data and no part of a graph's key, but this the executor looks at (a
// select against zero is a relu, executor.py:_masks_from_results): it asks here, and the key of a graph with a select says it of every number.
bool zero_number(PyObject* u) {
    PyObject *n = own(u, s_num), *h = n && PyLong_CheckExact(n) && PyLong_AsLongLong(n) == 1 && absent(u, s__op) ? own(u, s__host) : nullptr;
    Py_buffer view;
    if (!h || h == Py_None) return false;
    if (PyObject_GetBuffer(h, &view, PyBUF_SIMPLE)) { PyErr_Clear(); return false; }
    bool zero = view.len == view.itemsize;
    for (Py_ssize_t i = 0; zero && i < view.len; i++) zero = ((const char*)view.buf)[i] == 0;
    PyBuffer_Release(&view);
    return zero;
}
PyObject* py_zero_number(PyObject*, PyObject* u) { return PyBool_FromLong(zero_number(u)); }

// signature(ops, targets, flags): everything the execution of `ops` depends on besides the data, as bytes (with what ops of other classes
// say of themselves beside them), or None where an op does not know or its result is gone.
PyObject* py_signature(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    if (nargs != 3 || !PyList_Check(args[0]) || !PyList_Check(args[1]) || !PyDict_Check(args[2])) return PyErr_Format(PyExc_TypeError, "signature(ops, targets, flags)");
    std::unordered_map<PyObject*, int> made, leaf;
    std::unordered_set<PyObject*> targets;
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(args[1]); i++) targets.insert(PyList_GET_ITEM(args[1], i));
    std::vector<PyObject*> leaves;
    bool selects = false;
    Key k;
    k.b.reserve(4096);
    Ref others;
    const Py_ssize_t n = PyList_GET_SIZE(args[0]);
    k.num(n);
    for (Py_ssize_t i = 0; i < n; i++) {
        PyObject* op = PyList_GET_ITEM(args[0], i);
        PyTypeObject* t = Py_TYPE(op);
        PyObject* ref = own(op, s__out_ref);
        PyObject* out = ref && ref != Py_None ? PyWeakref_GetObject(ref) : nullptr;
        if (!out || out == Py_None) Py_RETURN_NONE;
        bool ok = true;
        auto get = [&](PyObject* name) { return own(op, name); };
        if (t == t_unary) { k.b.push_back('u'); ok = k.text(get(s_op)); }
        else if (t == t_binary) { k.b.push_back('b'); ok = k.text(get(s_op)); }
        else if (t == t_ternary) { k.b.push_back('t'); selects = true; }
        else if (t == t_broadcast) { k.b.push_back('c'); ok = k.integer(get(s_bcast_mask)) && k.integer(get(s_keepdims_mask)); }
        else if (t == t_reduce) { k.b.push_back('r'); ok = k.text(get(s_op)) && k.integer(get(s_reduce_mask)) && k.integer(get(s_keepdims_mask)); }
        else if (t == t_reindex) {
            k.b.push_back('x');
            PyObject* ov = get(s_overflow_value);
            const double o = ov ? PyFloat_AsDouble(ov) : 0.0;
            k.b.append((const char*)&o, sizeof o);
            k.b.push_back(flag(op, s_same_memory) ? 1 : 0);
            ok = !PyErr_Occurred() && k.texts(get(s_indexes)) && k.texts(get(s_overflow_conditions));
        } else if (t == t_reindex_reduce) { k.b.push_back('s'); ok = k.text(get(s_op)) && k.texts(get(s_indexes)) && k.texts(get(s_overflow_conditions)); }
        else {
            Ref s(PyObject_CallMethodNoArgs(op, s_sig));
            if (!s) return nullptr;
            if (s.p == Py_None) Py_RETURN_NONE;
            if (!others) others = Ref(PyList_New(0));
            if (!others || PyList_Append(others.p, s.p)) return nullptr;
            k.b.push_back('o');
        }
        if (!ok || !k.var(out)) return nullptr;
        k.b.push_back((char)((targets.count(out) ? 1 : 0) | (absent(out, s__buf) ? 2 : 0) | (flag(out, s__stop_fuse) ? 4 : 0)));
        PyObject* ins = own(op, s_inputs);
        if (!ins || !PyList_Check(ins)) return PyErr_Format(PyExc_TypeError, "an op's inputs are a list");
        k.num(PyList_GET_SIZE(ins));
        for (Py_ssize_t j = 0; j < PyList_GET_SIZE(ins); j++) {
            PyObject* u = PyList_GET_ITEM(ins, j);
            auto it = made.find(u);
            if (it != made.end()) {
                k.num(it->second);
                continue;
            }
            auto [l, first] = leaf.emplace(u, (int)leaf.size());
            k.num(-1 - l->second);
            if (first) {
                leaves.push_back(u);
                if (!k.var(u)) return nullptr;
                k.b.push_back((char)((absent(u, s__op) ? 1 : 0) | (absent(u, s__buf) ? 2 : 0) | (absent(u, s__host) ? 4 : 0) | (flag(u, s__stop_fuse) ? 8 : 0)));
            }
        }
        made[out] = (int)i;
    }
    if (selects)
        for (PyObject* u : leaves) k.b.push_back(zero_number(u) ? 1 : 0);
    // the flags are entered once and keep their order
    PyObject *name, *value;
    Py_ssize_t at = 0;
    while (PyDict_Next(args[2], &at, &name, &value)) {
        if (PyBool_Check(value)) k.b.push_back(value == Py_True ? 1 : 0);
        else {
            Ref s(PyObject_Str(value));
            if (!s) return nullptr;
            k.b.push_back(2);
            if (!k.text(s.p)) return nullptr;
        }
    }
    long long amp;
    if (amp_now(&amp)) return nullptr;
    k.num(amp);
    Ref bytes(PyBytes_FromStringAndSize(k.b.data(), (Py_ssize_t)k.b.size()));
    if (!bytes || !others) return bytes.give();
    Ref rest(PyList_AsTuple(others.p));
    return rest ? PyTuple_Pack(2, bytes.p, rest.p) : nullptr;
}

PyObject* py_as_var(PyObject*, PyObject* v) { return as_var(v); }

PyObject* py_setup(PyObject*, PyObject* ns) {
    struct { const char* name; PyObject** to; } want[] = {
        {"Var", (PyObject**)&t_var}, {"UnaryOp", (PyObject**)&t_unary}, {"BinaryOp", (PyObject**)&t_binary}, {"TernaryOp", (PyObject**)&t_ternary},
        {"BroadcastOp", (PyObject**)&t_broadcast}, {"ReduceOp", (PyObject**)&t_reduce}, {"ReindexOp", (PyObject**)&t_reindex}, {"ReindexReduceOp", (PyObject**)&t_reindex_reduce},
        {"_flags", &g_flags}, {"dt", &g_dt}, {"_grad_enabled", &g_grad_enabled}, {"array", &g_array}, {"_array_like", &g_as_var}, {"_scalar_vars", &g_scalars},
        {"_DTYPE_SET", &g_dtypes}, {"_UNARY_SET", &g_unary_ops}, {"_BINARY_SET", &g_binary_ops}, {"_REDUCE_SET", &g_reduce_ops}};
    for (auto& w : want) {
        PyObject* v = PyDict_GetItemString(ns, w.name);
        if (!v) return PyErr_Format(PyExc_KeyError, "setup: %s", w.name);
        PyObject* old = *w.to;
        *w.to = keep(v);
        Py_XDECREF(old);
    }
    PyObject* m = PyDict_GetItemString(ns, "_MAX_DIM");
    if (!m) return PyErr_Format(PyExc_KeyError, "setup: _MAX_DIM");
    g_max_dim = PyLong_AsLongLong(m);
    Py_RETURN_NONE;
}

#define FAST(name, doc) {#name, (PyCFunction)(void (*)(void))py_##name, METH_FASTCALL | METH_KEYWORDS, doc}
PyMethodDef methods[] = {
    FAST(unary, "unary(x, op, force_dtype=None, allow_forward=True): ops/unary_op.cc:860-889.  `op` is a unary op name or a dtype name."),
    FAST(binary, "binary(x, y, op): ops/binary_op.cc:421-474: broadcasts are inserted when ranks differ or an extent is 1 on one side only; other mismatches are errors."),
    FAST(ternary, "ternary(cond, x, y): ops/ternary_op.cc:21-47."),
    FAST(broadcast, "broadcast(x, shape, dims=()) / broadcast(x, y, dims): `dims` name the new axes of the output, the other axes align right to left (ops/broadcast_to_op.cc:23-96)."),
    FAST(broadcast_mask, "make_broadcast_to(x, shape, dims_mask, keepdims_mask), used by gradients."),
    FAST(reduce, "reduce(x, op, dims=(), keepdims=False): ops/reduce_op.cc:257-337."),
    FAST(reduce_mask, "reduce by masks of reduced and of kept axes."),
    FAST(make_number, "make_number(value, like): ops/op_utils.cc:19-36: a [1] array of like's dtype broadcast to like."),
    {"as_var", py_as_var, METH_O, "a Var, or the Var of a number or array"},
    {"new_id", py_new_id, METH_NOARGS, "the next id of a Var or op"},
    {"pending_ops", py_pending_ops, METH_O, "pending producers behind the targets, in topological order"},
    {"zero_number", py_zero_number, METH_O, "zero_number(var): whether it is one element in host memory whose bytes are all zero"},
    {"signature", (PyCFunction)(void (*)(void))py_signature, METH_FASTCALL, "signature(ops, targets, flags): hashable description of a graph, or None"},
    {"gradients", (PyCFunction)(void (*)(void))py_gradients, METH_FASTCALL, "gradients(loss, targets, others): a gradient per target"},
    {"setup", py_setup, METH_O, "takes the classes and tables of core.py"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_graph", "Graph building of the front end.", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__graph(void) {
#define INTERN(n) if (!(s_##n = PyUnicode_InternFromString(#n))) return nullptr;
    NAMES(INTERN)
#undef INTERN
    struct { PyObject** to; const char* text; } more[] = {{&s_void, "void"}, {&s_multiply, "multiply"}, {&s_divide, "divide"}, {&s_subtract, "subtract"}, {&s_negative, "negative"}, {&s_equal, "equal"}};
    for (auto& m : more)
        if (!(*m.to = PyUnicode_InternFromString(m.text))) return nullptr;
    return PyModule_Create(&module);
}
