// pyeval.cpp — the front end's expression trees as xg_expr descriptors, and
// the evaluation calls on them, for CPython.
//
// core.py builds trees of Func / Scalar / DeviceArray / IndexView / Reducer
// objects.  pack(root, reducer_fn) walks one tree once and lays out its nodes,
// leaves and constants as the C ABI wants them (arguments before users, an
// object used twice becomes one node or leaf); the Packed object's methods
// call the library with them.  Doing this through ctypes structures cost more
// than everything else in a small call: an eager c = a * b + exp(-a * a) of
// [32, 96] took 24.7 us a call, of which the kernel is 3.5 us.
//
// A Packed object lives for one call: nothing is kept between calls.  The
// library runs without the GIL; its status goes back to core.py, which maps it
// to an exception.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstring>
#include <new>
#include <vector>

#include "xg.h"

namespace {

// the classes of core.py (setup()), and interned attribute names
PyObject *c_array, *c_placeholder, *c_func, *c_scalar, *c_reducer, *c_index;
PyObject *s_storage, *s_data_ptr, *s_is_cuda, *s_dtype_code, *s_shape, *s_strides, *s_offset, *s_op, *s_args, *s_index,
    *s_value, *s_offsets, *s_source, *s_axes, *s_keep_dims, *s_initial, *s_acc_dtype, *s_ddof, *s_immediate,
    *s_to_abi;

struct Ref {  // an owned reference
    PyObject* p;
    explicit Ref(PyObject* o) : p(o) {}
    Ref(const Ref&) = delete;
    ~Ref() { Py_XDECREF(p); }
    explicit operator bool() const { return p != nullptr; }
};

bool is_a(PyObject* o, PyObject* cls) {
    if (reinterpret_cast<PyObject*>(Py_TYPE(o)) == cls) return true;
    return PyType_IsSubtype(Py_TYPE(o), reinterpret_cast<PyTypeObject*>(cls)) != 0;
}

bool int_of(PyObject* o, long long* v) {
    *v = PyLong_AsLongLong(o);
    return !(*v == -1 && PyErr_Occurred());
}

bool int_attr(PyObject* o, PyObject* name, long long* v) {
    Ref a(PyObject_GetAttr(o, name));
    return a && int_of(a.p, v);
}

// a DeviceArray (or anything with to_abi()) as an xg_tensor; *cuda is cleared
// when a device array's storage is not on the GPU
bool tensor_of(PyObject* a, xg_tensor* t, bool* cuda) {
    std::memset(t, 0, sizeof *t);
    const bool plain = reinterpret_cast<PyObject*>(Py_TYPE(a)) == c_array;
    const bool stand_in = is_a(a, c_placeholder);
    if (!plain && !stand_in) {
        if (is_a(a, c_array)) {
            Ref st(PyObject_GetAttr(a, s_storage));
            if (!st) return false;
            Ref c(PyObject_GetAttr(st.p, s_is_cuda));
            if (!c) PyErr_Clear();
            if (!c || PyObject_IsTrue(c.p) != 1) *cuda = false;
        }
        Ref abi(PyObject_CallMethodNoArgs(a, s_to_abi));
        if (!abi) return false;
        Py_buffer b;
        if (PyObject_GetBuffer(abi.p, &b, PyBUF_SIMPLE) != 0) return false;
        const bool ok = b.len == Py_ssize_t(sizeof *t);
        if (ok) std::memcpy(t, b.buf, sizeof *t);
        PyBuffer_Release(&b);
        if (!ok) PyErr_SetString(PyExc_TypeError, "not a tensor descriptor");
        return ok;
    }
    Ref st(PyObject_GetAttr(a, s_storage));
    if (!st) return false;
    if (!stand_in) {
        Ref c(PyObject_GetAttr(st.p, s_is_cuda));
        if (!c) PyErr_Clear();
        if (!c || PyObject_IsTrue(c.p) != 1) *cuda = false;
    }
    Ref ptr(PyObject_CallMethodNoArgs(st.p, s_data_ptr));
    if (!ptr) return false;
    t->data = PyLong_AsVoidPtr(ptr.p);
    if (PyErr_Occurred()) return false;
    long long v = 0;
    if (!int_attr(a, s_dtype_code, &v)) return false;
    t->dtype = int32_t(v);
    if (!int_attr(a, s_offset, &v)) return false;
    t->offset = v;
    Ref shape(PyObject_GetAttr(a, s_shape)), strides(PyObject_GetAttr(a, s_strides));
    if (!shape || !strides) return false;
    if (!PyTuple_Check(shape.p) || !PyTuple_Check(strides.p)) {
        PyErr_SetString(PyExc_TypeError, "an array's shape and strides are tuples");
        return false;
    }
    const Py_ssize_t n = PyTuple_GET_SIZE(shape.p);
    if (n > XG_MAX_RANK) {
        PyErr_SetString(PyExc_IndexError, "invalid index");
        return false;
    }
    t->ndim = int32_t(n);
    const Py_ssize_t m = PyTuple_GET_SIZE(strides.p) < n ? PyTuple_GET_SIZE(strides.p) : n;
    for (Py_ssize_t k = 0; k < m; ++k) {
        if (!int_of(PyTuple_GET_ITEM(shape.p, k), &v)) return false;
        t->shape[k] = v;
        if (!int_of(PyTuple_GET_ITEM(strides.p, k), &v)) return false;
        t->strides[k] = v;
    }
    return true;
}

// core.Scalar -> xg_scalar: floats as double, integers by their low 64 bits
bool scalar_of(PyObject* o, xg_scalar* s) {
    std::memset(s, 0, sizeof *s);
    long long dt = 0;
    if (!int_attr(o, s_dtype_code, &dt)) return false;
    s->dtype = int32_t(dt);
    Ref v(PyObject_GetAttr(o, s_value));
    if (!v) return false;
    if (dt == XG_FLOAT32 || dt == XG_FLOAT64) {
        Ref f(PyNumber_Float(v.p));
        if (!f) return false;
        s->v.f = PyFloat_AS_DOUBLE(f.p);
    } else {
        Ref i(PyNumber_Long(v.p));
        if (!i) return false;
        s->v.u = PyLong_AsUnsignedLongLongMask(i.p);
        if (PyErr_Occurred()) return false;
    }
    return true;
}

struct Packed {
    PyObject_HEAD
    std::vector<xg_node>* nodes;
    std::vector<xg_tensor>* leaves;
    std::vector<xg_scalar>* consts;
    std::vector<PyObject*>* keep;  // owned: the root and the evaluated reducers
    xg_expr e;
    bool cuda;  // every device array read is on the GPU
};

struct Walk {
    Packed* p;
    PyObject* reducer_fn;
    struct Seen { PyObject* o; int32_t node; };
    std::vector<Seen> seen;       // visited objects (alive through the root) and their nodes
    std::vector<PyObject*> slots; // leaf objects in slot order

    int32_t add(int32_t op, int nargs, const int32_t* args, int32_t index) {
        xg_node n{};
        n.op = op;
        n.nargs = nargs;
        for (int k = 0; k < nargs; ++k) n.args[k] = args[k];
        n.index = index;
        p->nodes->push_back(n);
        if (p->nodes->size() > XG_MAX_NODES) {
            PyErr_SetString(PyExc_NotImplementedError, "expression has too many nodes");
            return -1;
        }
        return int32_t(p->nodes->size()) - 1;
    }

    int32_t slot(PyObject* a) {
        for (size_t k = 0; k < slots.size(); ++k)
            if (slots[k] == a) return int32_t(k);
        xg_tensor t;
        if (!tensor_of(a, &t, &p->cuda)) return -1;
        slots.push_back(a);
        p->leaves->push_back(t);
        return int32_t(slots.size()) - 1;
    }

    int32_t visit(PyObject* o) {
        for (const Seen& s : seen)
            if (s.o == o) return s.node;
        const int32_t r = visit_new(o);
        if (r >= 0) seen.push_back(Seen{o, r});
        return r;
    }

    int32_t visit_new(PyObject* o) {
        if (is_a(o, c_array)) {
            const int32_t s = slot(o);
            return s < 0 ? -1 : add(XG_OP_LEAF, 0, nullptr, s);
        }
        if (is_a(o, c_func)) {
            Ref args(PyObject_GetAttr(o, s_args));
            if (!args) return -1;
            if (!PyTuple_Check(args.p)) {
                PyErr_SetString(PyExc_TypeError, "a node's arguments are a tuple");
                return -1;
            }
            const Py_ssize_t n = PyTuple_GET_SIZE(args.p);
            if (n > 3) {
                PyErr_SetString(PyExc_IndexError, "invalid index");
                return -1;
            }
            int32_t a[3] = {0, 0, 0};
            if (Py_EnterRecursiveCall(" in an expression")) return -1;
            for (Py_ssize_t k = 0; k < n; ++k) {
                a[k] = visit(PyTuple_GET_ITEM(args.p, k));
                if (a[k] < 0) break;
            }
            Py_LeaveRecursiveCall();
            for (Py_ssize_t k = 0; k < n; ++k)
                if (a[k] < 0) return -1;
            long long op = 0, index = 0;
            if (!int_attr(o, s_op, &op) || !int_attr(o, s_index, &index)) return -1;
            return add(int32_t(op), int(n), a, int32_t(index));
        }
        if (is_a(o, c_scalar)) {
            xg_scalar s;
            if (!scalar_of(o, &s)) return -1;
            p->consts->push_back(s);
            return add(XG_OP_CONST, 0, nullptr, int32_t(p->consts->size()) - 1);
        }
        if (is_a(o, c_index)) {  // a gather of the source at the offsets' values
            Ref off(PyObject_GetAttr(o, s_offsets)), src(PyObject_GetAttr(o, s_source));
            if (!off || !src) return -1;
            if (Py_EnterRecursiveCall(" in an expression")) return -1;
            const int32_t a = visit(off.p);
            Py_LeaveRecursiveCall();
            if (a < 0) return -1;
            const int32_t s = slot(src.p);
            return s < 0 ? -1 : add(XG_OP_GATHER, 1, &a, s);
        }
        if (is_a(o, c_reducer)) {  // evaluated first; its value is a leaf
            if (reducer_fn == Py_None) {
                PyErr_SetString(PyExc_RuntimeError, "reducer inside an expression needs an evaluation context");
                return -1;
            }
            PyObject* tmp = PyObject_CallOneArg(reducer_fn, o);
            if (!tmp) return -1;
            p->keep->push_back(tmp);
            const int32_t s = slot(tmp);
            return s < 0 ? -1 : add(XG_OP_LEAF, 0, nullptr, s);
        }
        PyErr_Format(PyExc_TypeError, "not an expression: %R", o);
        return -1;
    }
};

void packed_dealloc(PyObject* self) {
    Packed* p = reinterpret_cast<Packed*>(self);
    delete p->nodes;
    delete p->leaves;
    delete p->consts;
    if (p->keep)
        for (PyObject* o : *p->keep) Py_XDECREF(o);
    delete p->keep;
    Py_TYPE(self)->tp_free(self);
}

extern PyTypeObject packed_type;

PyObject* py_pack(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 2) {
        PyErr_SetString(PyExc_TypeError, "pack(root, reducer_fn)");
        return nullptr;
    }
    Packed* p = reinterpret_cast<Packed*>(packed_type.tp_alloc(&packed_type, 0));
    if (!p) return nullptr;
    Ref own(reinterpret_cast<PyObject*>(p));
    try {
        p->nodes = new std::vector<xg_node>;
        p->leaves = new std::vector<xg_tensor>;
        p->consts = new std::vector<xg_scalar>;
        p->keep = new std::vector<PyObject*>;
        p->nodes->reserve(16);
        p->leaves->reserve(8);
        p->consts->reserve(8);
        p->cuda = true;
        Py_INCREF(a[0]);
        p->keep->push_back(a[0]);
        Walk w{p, a[1], {}, {}};
        w.seen.reserve(16);
        w.slots.reserve(8);
        if (w.visit(a[0]) < 0) return nullptr;
    } catch (const std::bad_alloc&) {
        return PyErr_NoMemory();
    }
    p->e = xg_expr{};
    p->e.n_nodes = int32_t(p->nodes->size());
    p->e.n_leaves = int32_t(p->leaves->size());
    p->e.n_consts = int32_t(p->consts->size());
    p->e.nodes = p->nodes->data();
    p->e.leaves = p->leaves->data();
    p->e.consts = p->consts->data();
    Py_INCREF(own.p);
    return own.p;
}

// core.Reducer -> xg_reduce_desc
bool reduce_of(PyObject* r, xg_reduce_desc* d) {
    std::memset(d, 0, sizeof *d);
    long long v = 0;
    if (!int_attr(r, s_op, &v)) return false;
    d->op = int32_t(v);
    if (!int_attr(r, s_acc_dtype, &v)) return false;
    d->acc_dtype = int32_t(v);
    Ref axes(PyObject_GetAttr(r, s_axes));
    if (!axes) return false;
    if (axes.p == Py_None) {
        d->n_axes = -1;
    } else {
        if (!PyList_Check(axes.p)) {
            PyErr_SetString(PyExc_TypeError, "a reducer's axes are a list");
            return false;
        }
        const Py_ssize_t n = PyList_GET_SIZE(axes.p);
        if (n > XG_MAX_RANK) {
            PyErr_SetString(PyExc_RuntimeError, "too many axes");
            return false;
        }
        d->n_axes = int32_t(n);
        for (Py_ssize_t k = 0; k < n; ++k) {
            if (!int_of(PyList_GET_ITEM(axes.p, k), &v)) return false;
            d->axes[k] = int32_t(v);
        }
    }
    if (!int_attr(r, s_keep_dims, &v)) return false;
    d->keep_dims = int32_t(v);
    Ref init(PyObject_GetAttr(r, s_initial));
    if (!init) return false;
    if (init.p != Py_None) {
        if (!is_a(init.p, c_scalar)) {
            PyErr_SetString(PyExc_TypeError, "a reduction's initial value is a scalar");
            return false;
        }
        d->has_initial = 1;
        if (!scalar_of(init.p, &d->initial)) return false;
    }
    if (!int_attr(r, s_ddof, &v)) return false;
    d->ddof = int32_t(v);
    Ref imm(PyObject_GetAttr(r, s_immediate));
    if (!imm) return false;
    const int on = PyObject_IsTrue(imm.p);
    if (on < 0) return false;
    d->flags = on ? XG_REDUCE_IMMEDIATE : 0;
    return true;
}

bool on_gpu(bool cuda) {
    if (!cuda) PyErr_SetString(PyExc_RuntimeError, "evaluation needs device (cuda) arrays");
    return cuda;
}

// (dtype code, shape) or the library's status
PyObject* info_result(int st, int32_t dt, int32_t nd, const int64_t* shape) {
    if (st != XG_OK) return PyLong_FromLong(st);
    Ref shp(PyTuple_New(nd));
    if (!shp) return nullptr;
    for (int32_t k = 0; k < nd; ++k) {
        PyObject* v = PyLong_FromLongLong(shape[k]);
        if (!v) return nullptr;
        PyTuple_SET_ITEM(shp.p, k, v);
    }
    return Py_BuildValue("(iO)", int(dt), shp.p);
}

PyObject* m_info(PyObject* self, PyObject*) {
    Packed* p = reinterpret_cast<Packed*>(self);
    int32_t dt = 0, nd = 0;
    int64_t shape[XG_MAX_RANK];
    const int st = xg_expr_info(&p->e, &dt, &nd, shape);
    return info_result(st, dt, nd, shape);
}

// the descriptor's bytes, for comparison with core.serialize()
PyObject* m_raw(PyObject* self, PyObject*) {
    Packed* p = reinterpret_cast<Packed*>(self);
    auto bytes = [](const void* d, size_t n) { return PyBytes_FromStringAndSize(static_cast<const char*>(d), Py_ssize_t(n)); };
    Ref a(bytes(p->nodes->data(), p->nodes->size() * sizeof(xg_node)));
    Ref b(bytes(p->leaves->data(), p->leaves->size() * sizeof(xg_tensor)));
    Ref c(bytes(p->consts->data(), p->consts->size() * sizeof(xg_scalar)));
    if (!a || !b || !c) return nullptr;
    return PyTuple_Pack(3, a.p, b.p, c.p);
}

PyObject* m_reduce_info(PyObject* self, PyObject* r) {
    Packed* p = reinterpret_cast<Packed*>(self);
    xg_reduce_desc d;
    if (!reduce_of(r, &d)) return nullptr;
    int32_t dt = 0, nd = 0;
    int64_t shape[XG_MAX_RANK];
    const int st = xg_reduce_info(&p->e, &d, &dt, &nd, shape);
    return info_result(st, dt, nd, shape);
}

bool scan_args(PyObject* const* a, xg_scan_desc* d) {
    long long op, acc, axis;
    if (!int_of(a[0], &op) || !int_of(a[1], &acc) || !int_of(a[2], &axis)) return false;
    std::memset(d, 0, sizeof *d);
    d->op = int32_t(op);
    d->acc_dtype = int32_t(acc);
    d->axis = int32_t(axis);
    return true;
}

PyObject* m_scan_info(PyObject* self, PyObject* const* a, Py_ssize_t n) {
    Packed* p = reinterpret_cast<Packed*>(self);
    xg_scan_desc d;
    if (n != 3) {
        PyErr_SetString(PyExc_TypeError, "scan_info(op, dtype, axis)");
        return nullptr;
    }
    if (!scan_args(a, &d)) return nullptr;
    int32_t dt = 0, nd = 0;
    int64_t shape[XG_MAX_RANK];
    const int st = xg_scan_info(&p->e, &d, &dt, &nd, shape);
    return info_result(st, dt, nd, shape);
}

// the output's descriptor and the stream of an evaluation: its address, or a
// function to ask for it (only once all arrays are known to be on the GPU:
// without one torch has no stream to give)
bool target(Packed* p, PyObject* out, PyObject* stream, xg_tensor* t, xg_stream_t* st) {
    bool cuda = p->cuda;
    if (!tensor_of(out, t, &cuda) || !on_gpu(cuda)) return false;
    Ref asked(PyLong_Check(stream) ? nullptr : PyObject_CallNoArgs(stream));
    if (!asked && !PyLong_Check(stream)) return false;
    *st = reinterpret_cast<xg_stream_t>(PyLong_AsVoidPtr(asked ? asked.p : stream));
    return !PyErr_Occurred();
}

PyObject* m_assign(PyObject* self, PyObject* const* a, Py_ssize_t n) {  // (out, stream)
    Packed* p = reinterpret_cast<Packed*>(self);
    xg_tensor t;
    xg_stream_t st;
    if (n != 2) {
        PyErr_SetString(PyExc_TypeError, "assign(out, stream)");
        return nullptr;
    }
    if (!target(p, a[0], a[1], &t, &st)) return nullptr;
    int r;
    Py_BEGIN_ALLOW_THREADS
    r = xg_assign(&p->e, &t, st);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(r);
}

PyObject* m_reduce(PyObject* self, PyObject* const* a, Py_ssize_t n) {  // (reducer, out, stream)
    Packed* p = reinterpret_cast<Packed*>(self);
    xg_tensor t;
    xg_stream_t st;
    xg_reduce_desc d;
    if (n != 3) {
        PyErr_SetString(PyExc_TypeError, "reduce(reducer, out, stream)");
        return nullptr;
    }
    if (!reduce_of(a[0], &d) || !target(p, a[1], a[2], &t, &st)) return nullptr;
    int r;
    Py_BEGIN_ALLOW_THREADS
    r = xg_reduce(&p->e, &d, &t, st);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(r);
}

PyObject* m_scan(PyObject* self, PyObject* const* a, Py_ssize_t n) {  // (op, dtype, axis, out, stream)
    Packed* p = reinterpret_cast<Packed*>(self);
    xg_tensor t;
    xg_stream_t st;
    xg_scan_desc d;
    if (n != 5) {
        PyErr_SetString(PyExc_TypeError, "scan(op, dtype, axis, out, stream)");
        return nullptr;
    }
    if (!scan_args(a, &d) || !target(p, a[3], a[4], &t, &st)) return nullptr;
    int r;
    Py_BEGIN_ALLOW_THREADS
    r = xg_scan(&p->e, &d, &t, st);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(r);
}

PyObject* m_argwhere_mark(PyObject* self, PyObject* const* a, Py_ssize_t n) {  // (order, buffer, stream)
    Packed* p = reinterpret_cast<Packed*>(self);
    long long order = 0;
    if (n != 3) {
        PyErr_SetString(PyExc_TypeError, "argwhere_mark(order, buffer, stream)");
        return nullptr;
    }
    if (!int_of(a[0], &order) || !on_gpu(p->cuda)) return nullptr;
    void* buf = PyLong_AsVoidPtr(a[1]);
    xg_stream_t st = reinterpret_cast<xg_stream_t>(PyLong_AsVoidPtr(a[2]));
    if (PyErr_Occurred()) return nullptr;
    int r;
    Py_BEGIN_ALLOW_THREADS
    r = xg_argwhere_mark(&p->e, int32_t(order), buf, st);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(r);
}

PyObject* m_argwhere_list(PyObject* self, PyObject* const* a, Py_ssize_t n) {  // (order, buffer, out, stream)
    Packed* p = reinterpret_cast<Packed*>(self);
    xg_tensor t;
    xg_stream_t st;
    long long order = 0;
    if (n != 4) {
        PyErr_SetString(PyExc_TypeError, "argwhere_list(order, buffer, out, stream)");
        return nullptr;
    }
    if (!int_of(a[0], &order) || !target(p, a[2], a[3], &t, &st)) return nullptr;
    void* buf = PyLong_AsVoidPtr(a[1]);
    if (PyErr_Occurred()) return nullptr;
    int r;
    Py_BEGIN_ALLOW_THREADS
    r = xg_argwhere_list(&p->e, int32_t(order), buf, &t, st);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(r);
}

#define XG_FAST(f) reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f))
PyMethodDef packed_methods[] = {
    {"info", m_info, METH_NOARGS, "(dtype code, shape) or a status"},
    {"raw", m_raw, METH_NOARGS, "the bytes of the nodes, leaves and constants"},
    {"reduce_info", m_reduce_info, METH_O, "(dtype code, shape) of a reducer's result, or a status"},
    {"scan_info", XG_FAST(m_scan_info), METH_FASTCALL, "(dtype code, shape) of a scan's result, or a status"},
    {"assign", XG_FAST(m_assign), METH_FASTCALL, "xg_assign(out, stream)"},
    {"reduce", XG_FAST(m_reduce), METH_FASTCALL, "xg_reduce(reducer, out, stream)"},
    {"scan", XG_FAST(m_scan), METH_FASTCALL, "xg_scan(op, dtype, axis, out, stream)"},
    {"argwhere_mark", XG_FAST(m_argwhere_mark), METH_FASTCALL, "xg_argwhere_mark(order, buffer, stream)"},
    {"argwhere_list", XG_FAST(m_argwhere_list), METH_FASTCALL, "xg_argwhere_list(order, buffer, out, stream)"},
    {nullptr, nullptr, 0, nullptr}};

PyTypeObject packed_type = [] {
    PyTypeObject t{PyVarObject_HEAD_INIT(nullptr, 0)};
    t.tp_name = "_xgpy.Packed";
    t.tp_basicsize = sizeof(Packed);
    t.tp_dealloc = packed_dealloc;
    t.tp_flags = Py_TPFLAGS_DEFAULT;
    t.tp_methods = packed_methods;
    return t;
}();

PyObject* py_setup(PyObject*, PyObject* a) {
    PyObject** dst[] = {&c_array, &c_placeholder, &c_func, &c_scalar, &c_reducer, &c_index};
    constexpr Py_ssize_t n = sizeof dst / sizeof *dst;
    if (!PyTuple_Check(a) || PyTuple_GET_SIZE(a) != n) {
        PyErr_SetString(PyExc_TypeError, "setup(DeviceArray, placeholder, Func, Scalar, Reducer, IndexView)");
        return nullptr;
    }
    for (Py_ssize_t k = 0; k < n; ++k) {
        PyObject* c = PyTuple_GET_ITEM(a, k);
        if (!PyType_Check(c)) {
            PyErr_SetString(PyExc_TypeError, "setup() takes classes");
            return nullptr;
        }
        Py_INCREF(c);
        Py_XDECREF(*dst[k]);
        *dst[k] = c;
    }
    Py_RETURN_NONE;
}

PyMethodDef module_methods[] = {
    {"setup", py_setup, METH_O, "the front end's classes"},
    {"pack", XG_FAST(py_pack), METH_FASTCALL, "pack(root, reducer_fn): an expression tree as a descriptor"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_xgpy", "expression trees as xg_expr descriptors", -1,
                          module_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__xgpy(void) {
    const struct { PyObject** s; const char* n; } names[] = {
        {&s_storage, "storage"}, {&s_data_ptr, "data_ptr"}, {&s_is_cuda, "is_cuda"}, {&s_dtype_code, "dtype_code"},
        {&s_shape, "_shape"}, {&s_strides, "strides"}, {&s_offset, "offset"}, {&s_op, "op"}, {&s_args, "args"},
        {&s_index, "index"}, {&s_value, "value"}, {&s_offsets, "offsets"}, {&s_source, "source"},
        {&s_axes, "axes"}, {&s_keep_dims, "keep_dims"}, {&s_initial, "initial"}, {&s_acc_dtype, "acc_dtype"},
        {&s_ddof, "ddof"}, {&s_immediate, "immediate"}, {&s_to_abi, "to_abi"}};
    for (const auto& n : names) {
        *n.s = PyUnicode_InternFromString(n.n);
        if (!*n.s) return nullptr;
    }
    if (PyType_Ready(&packed_type) < 0) return nullptr;
    return PyModule_Create(&module_def);
}
