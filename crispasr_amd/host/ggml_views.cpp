// The host path of crispasr_amd/ggml.py in native code: the tensor views and the launching calls.
//
// A decoder step is a few hundred views and calls of a few microseconds of GPU work each, so what the host spends per
// call is what such a step costs.  In Python (ctypes descriptors, a stream object per call) it was 7.6 us for a copy, 9.3
// for an attention call and 2.9 per view, of which the library and the HIP launch are 2.9 and 4.7; here a call adds 0.5 us
// to those and a view costs 0.15.
//
// The module holds no pointer of its own to the library: ggml.lib() loads it (or an alternative build of it) and hands
// the entry points' addresses to bind().
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <stddef.h>
#include <stdint.h>
#include <string.h>

#include "../../include/mi355x_fattn.h"

namespace {

typedef int (*attn_fn)(const mi355x_tensor *, const mi355x_tensor *, const mi355x_tensor *, const mi355x_tensor *, const mi355x_tensor *,
                       const mi355x_fattn_params *, void *);

struct Bound {
    attn_fn flash_attn_ext, flash_attn_ext_noalloc;
    decltype(&mi355x_cpy) cpy;
    decltype(&mi355x_set_rows) set_rows;
    decltype(&mi355x_relpos_bias) relpos_bias;
    decltype(&mi355x_flash_attn_relpos) flash_attn_relpos;
    int (*get_device)(int *);
    int (*set_device)(int);
};
Bound g_lib;
PyObject * g_failed     = nullptr;      // called with a non-zero status: raises
PyObject * g_raw_stream = nullptr;      // device index -> handle of torch's current stream there
PyObject * g_host_buffer = nullptr;     // the HostBuffer class
PyObject * g_uint8 = nullptr, * g_int32 = nullptr, * g_int64 = nullptr;     // torch dtypes

PyObject * s_data_ptr, * s_numel, * s_get_device, * s_device, * s_index, * s_dtype, * s_dim, * s_is_contiguous, * s_cuda_stream,
         * s_shape, * s_element_size;

// bytes per element (or block of 32) of a storage type, 0 for one that is not known
int type_size(int t) {
    switch (t) {
        case MI355X_TYPE_F32:  return 4;
        case MI355X_TYPE_F16:  return 2;
        case MI355X_TYPE_Q4_0: return 18;
        case MI355X_TYPE_Q4_1: return 20;
        case MI355X_TYPE_Q5_0: return 22;
        case MI355X_TYPE_Q5_1: return 24;
        case MI355X_TYPE_Q8_0: return 34;
        default:               return 0;
    }
}
int block_size(int t) { return t == MI355X_TYPE_F32 || t == MI355X_TYPE_F16 ? 1 : 32; }

// ---- View: type, ne, nb and offset over a buffer ----------------------------------------------------------------

// The fields are ordinary attributes (buf, type, ne, nb, offset: entries of the instance's dict).  The C descriptor is made
// from them once, when a call first needs it.
struct View {
    PyObject_HEAD
    PyObject * dict;
    int        device;         // once resolved: the buffer's device index, -1 if it has none, or NO_BUFFER
    bool       resolved;
    mi355x_tensor t;
};
constexpr int NO_BUFFER = -2;
PyObject * s_buf, * s_type, * s_ne, * s_nb, * s_offset;

// int(x), wrapped to 64 bits as a ctypes field would
bool to_i64(PyObject * x, int64_t * out) {
    if (PyLong_CheckExact(x)) {
        *out = (int64_t)PyLong_AsUnsignedLongLongMask(x);
    } else {
        PyObject * n = PyNumber_Long(x);
        if (!n) return false;
        *out = (int64_t)PyLong_AsUnsignedLongLongMask(n);
        Py_DECREF(n);
    }
    return *out != -1 || !PyErr_Occurred();
}

// a tuple of ints from a sequence of numbers, filled up with ones to `fill` entries
PyObject * int_tuple(PyObject * seq, Py_ssize_t fill) {
    if (PyTuple_CheckExact(seq) && PyTuple_GET_SIZE(seq) >= fill) {
        Py_ssize_t i = 0;
        while (i < PyTuple_GET_SIZE(seq) && PyLong_CheckExact(PyTuple_GET_ITEM(seq, i))) i++;
        if (i == PyTuple_GET_SIZE(seq)) return Py_NewRef(seq);
    }
    PyObject * fast = PySequence_Fast(seq, "a sequence of numbers is needed");
    if (!fast) return nullptr;
    const Py_ssize_t n = PySequence_Fast_GET_SIZE(fast);
    PyObject * r = PyTuple_New(n > fill ? n : fill);
    for (Py_ssize_t i = 0; r && i < PyTuple_GET_SIZE(r); i++) {
        PyObject * x = i < n ? PyNumber_Long(PySequence_Fast_GET_ITEM(fast, i)) : PyLong_FromLong(1);
        if (!x) Py_CLEAR(r);
        else PyTuple_SET_ITEM(r, i, x);
    }
    Py_DECREF(fast);
    return r;
}

// up to 4 numbers of a sequence; their count, or -1
int ints_of(PyObject * seq, int64_t * out) {
    PyObject * fast = PySequence_Fast(seq, "a sequence of numbers is needed");
    if (!fast) return -1;
    Py_ssize_t n = PySequence_Fast_GET_SIZE(fast);
    if (n > 4) {
        PyErr_SetString(PyExc_ValueError, "at most 4 dimensions");
        n = -1;
    }
    for (Py_ssize_t i = 0; i < n; i++)
        if (!to_i64(PySequence_Fast_GET_ITEM(fast, i), &out[i])) n = -1;
    Py_DECREF(fast);
    return (int)n;
}

// contiguous strides, as a tuple
PyObject * contiguous_nb(int64_t type, PyObject * ne) {
    const int ts = type_size((int)type);
    int64_t e[4] = {1, 1, 1, 1};
    if (!ts) return PyErr_Format(PyExc_KeyError, "%lld", (long long)type);
    if (ints_of(ne, e) < 0) return nullptr;
    const int64_t bs = block_size((int)type), blocks = e[0] / bs - (e[0] % bs < 0 ? 1 : 0);
    const int64_t nb1 = ts * blocks, nb2 = (int64_t)((uint64_t)nb1 * (uint64_t)e[1]), nb3 = (int64_t)((uint64_t)nb2 * (uint64_t)e[2]);
    return Py_BuildValue("(iLLL)", ts, (long long)nb1, (long long)nb2, (long long)nb3);
}

// the fields of a fresh view; nb None: contiguous
bool view_fill(View * v, PyObject * buf, PyObject * type, PyObject * ne, PyObject * nb, PyObject * offset) {
    bool       ok  = false;
    int64_t    ti  = 0;
    PyObject * d   = PyDict_New();
    PyObject * ty  = PyNumber_Long(type);
    PyObject * ext = int_tuple(ne, 4);
    PyObject * str = nullptr;
    if (d && ty && ext && to_i64(ty, &ti)) {
        str = nb == Py_None ? contiguous_nb(ti, ext) : int_tuple(nb, 0);
        ok  = str && PyDict_SetItem(d, s_buf, buf) == 0 && PyDict_SetItem(d, s_type, ty) == 0 && PyDict_SetItem(d, s_ne, ext) == 0 &&
              PyDict_SetItem(d, s_nb, str) == 0 && PyDict_SetItem(d, s_offset, offset) == 0;
    }
    Py_XDECREF(ty);
    Py_XDECREF(ext);
    Py_XDECREF(str);
    if (!ok) {
        Py_XDECREF(d);
        return false;
    }
    Py_XSETREF(v->dict, d);
    v->resolved = false;
    return true;
}

PyObject * field(const View * v, PyObject * name) {         // borrowed
    PyObject * x = v->dict ? PyDict_GetItemWithError(v->dict, name) : nullptr;
    if (!x && !PyErr_Occurred()) PyErr_SetObject(PyExc_AttributeError, name);
    return x;
}

bool call_i64(PyObject * obj, PyObject * method, int64_t * out) {
    PyObject * r = PyObject_CallMethodNoArgs(obj, method);
    if (!r) return false;
    const bool ok = to_i64(r, out);
    Py_DECREF(r);
    return ok;
}

int view_init(View * v, PyObject * args, PyObject * kw) {
    static const char * names[] = {"buf", "type_", "ne", "nb", "offset", nullptr};
    PyObject * buf, * type, * ne, * nb = Py_None, * off = nullptr;
    if (!PyArg_ParseTupleAndKeywords(args, kw, "OOO|OO", (char **)names, &buf, &type, &ne, &nb, &off)) return -1;
    PyObject * o = off ? PyNumber_Long(off) : PyLong_FromLong(0);
    const bool ok = o && view_fill(v, buf, type, ne, nb, o);
    Py_XDECREF(o);
    if (!ok) return -1;
    if (buf == Py_None) return 0;
    const int host = g_host_buffer ? PyObject_IsInstance(buf, g_host_buffer) : 0;
    if (host) return host < 0 ? -1 : 0;
    PyObject * dt = PyObject_GetAttr(buf, s_dtype);
    if (!dt) return -1;
    Py_DECREF(dt);                                       // (a torch dtype lives as long as the interpreter)
    int64_t dim = 0, contiguous = 0;
    if (!call_i64(buf, s_dim, &dim) || !call_i64(buf, s_is_contiguous, &contiguous)) return -1;
    if (dt != g_uint8 || dim != 1 || !contiguous) {
        PyErr_SetString(PyExc_AssertionError, "a tensor's buffer is a contiguous 1-D uint8 tensor");
        return -1;
    }
    return 0;
}

int view_traverse(View * v, visitproc visit, void * arg) {
    Py_VISIT(v->dict);
    return 0;
}
int view_clear(View * v) {
    Py_CLEAR(v->dict);
    return 0;
}
void view_dealloc(View * v) {
    PyObject_GC_UnTrack(v);
    Py_XDECREF(v->dict);
    Py_TYPE(v)->tp_free((PyObject *)v);
}

// view(ne, nb, offset=0, type_=None): same buffer, new extents and strides, offset relative to this view
PyObject * view_view(View * self, PyObject * const * args, Py_ssize_t n, PyObject * kwnames) {
    PyObject * a[4] = {nullptr, nullptr, nullptr, nullptr};
    static const char * names[4] = {"ne", "nb", "offset", "type_"};
    if (n > 4) {
        PyErr_SetString(PyExc_TypeError, "view() takes at most 4 arguments");
        return nullptr;
    }
    for (Py_ssize_t i = 0; i < n; i++) a[i] = args[i];
    for (Py_ssize_t i = 0; kwnames && i < PyTuple_GET_SIZE(kwnames); i++) {
        PyObject * k = PyTuple_GET_ITEM(kwnames, i);
        int at = 0;
        while (at < 4 && PyUnicode_CompareWithASCIIString(k, names[at]) != 0) at++;
        if (at == 4 || a[at]) {
            PyErr_Format(PyExc_TypeError, "view(): unexpected argument %R", k);
            return nullptr;
        }
        a[at] = args[n + i];
    }
    if (!a[0] || !a[1]) {
        PyErr_SetString(PyExc_TypeError, "view() needs ne and nb");
        return nullptr;
    }
    PyObject * buf  = field(self, s_buf);
    PyObject * type = a[3] && a[3] != Py_None ? a[3] : field(self, s_type);
    PyObject * base = field(self, s_offset);
    if (!buf || !type || !base) return nullptr;
    PyObject * sum = a[2] ? PyNumber_Add(base, a[2]) : Py_NewRef(base);
    PyObject * off = sum ? PyNumber_Long(sum) : nullptr;
    Py_XDECREF(sum);
    View * v = off ? (View *)Py_TYPE(self)->tp_alloc(Py_TYPE(self), 0) : nullptr;
    if (v && !view_fill(v, buf, type, a[0], a[1], off)) Py_CLEAR(v);
    Py_XDECREF(off);
    return (PyObject *)v;
}

// the descriptor's fields (but for the address), and the offset
bool view_read(const View * v, mi355x_tensor * t, int64_t * offset) {
    PyObject * type = field(v, s_type), * ne = type ? field(v, s_ne) : nullptr, * nb = ne ? field(v, s_nb) : nullptr,
             * off = nb ? field(v, s_offset) : nullptr;
    int64_t x = 0, s[4] = {0, 0, 0, 0};
    memset(t, 0, sizeof(*t));
    if (!off || !to_i64(type, &x) || ints_of(ne, t->ne) < 0 || ints_of(nb, s) < 0 || !to_i64(off, offset)) return false;
    t->type = (int32_t)x;
    for (int i = 0; i < 4; i++) t->nb[i] = (size_t)s[i];
    return true;
}

// bytes from the first to one past the last byte of the view
bool span_bytes(const mi355x_tensor & t, __int128 * out) {
    const int ts = type_size(t.type);
    if (!ts) {
        PyErr_Format(PyExc_KeyError, "%d", (int)t.type);
        return false;
    }
    *out = 0;
    for (int i = 0; i < 4; i++)
        if (t.ne[i] == 0) return true;
    __int128 last = (__int128)(t.ne[0] / block_size(t.type) - 1) * (int64_t)t.nb[0];
    for (int i = 1; i < 4; i++) last += (__int128)(t.ne[i] - 1) * (int64_t)t.nb[i];
    *out = last + ts;
    return true;
}

void raise_status(int status, const char * message) {
    PyObject * r = g_failed ? PyObject_CallFunction(g_failed, "is", status, message) : nullptr;
    Py_XDECREF(r);
    if (!PyErr_Occurred()) PyErr_Format(PyExc_RuntimeError, "mi355x status %d", status);
}

// the address that the descriptor carries
bool view_address(const View * v, const mi355x_tensor & t, int64_t offset, int64_t * out) {
    PyObject * buf = field(v, s_buf);
    if (!buf) return false;
    if (buf == Py_None) {
        // planning before allocation: the predicates never dereference, they only look at the address's low bits
        // (buffers start on 256 bytes, so the view's offset modulo 256 stands for them)
        *out = ((offset % 256) + 256) % 256;
        return true;
    }
    __int128 span = 0;
    int64_t  size = 0, base = 0;
    if (!span_bytes(t, &span) || !call_i64(buf, s_numel, &size)) return false;
    if (offset + span > size) {
        raise_status(MI355X_ERR_INVALID, "tensor view exceeds its buffer");
        return false;
    }
    if (!call_i64(buf, s_data_ptr, &base)) return false;
    *out = base + offset;
    return true;
}

// the C descriptor and the device, once
bool view_resolve(View * v) {
    if (v->resolved) return true;
    mi355x_tensor t;
    int64_t offset = 0, p = 0, dev = NO_BUFFER;
    if (!view_read(v, &t, &offset) || !view_address(v, t, offset, &p)) return false;
    PyObject * buf = field(v, s_buf);
    if (buf != Py_None) {
        if (g_host_buffer && PyObject_TypeCheck(buf, (PyTypeObject *)g_host_buffer)) {
            PyObject * d = PyObject_GetAttr(buf, s_device);
            PyObject * i = d ? PyObject_GetAttr(d, s_index) : nullptr;
            Py_XDECREF(d);
            if (!i) return false;
            dev = -1;
            const bool ok = i == Py_None || to_i64(i, &dev);
            Py_DECREF(i);
            if (!ok) return false;
        } else if (!call_i64(buf, s_get_device, &dev)) {
            return false;
        }
    }
    t.data      = (void *)(uintptr_t)p;
    v->t        = t;
    v->device   = (int)dev;
    v->resolved = true;
    return true;
}

PyObject * view_span(View * v, PyObject *) {
    mi355x_tensor t;
    int64_t  off = 0;
    __int128 s = 0;
    if (!view_read(v, &t, &off) || !span_bytes(t, &s)) return nullptr;
    return PyLong_FromLongLong((long long)s);
}

PyObject * view_data_ptr(View * v, PyObject *) {
    mi355x_tensor t;
    int64_t off = 0, p = 0;
    if (!view_read(v, &t, &off) || !view_address(v, t, off, &p)) return nullptr;
    return PyLong_FromUnsignedLongLong((unsigned long long)p);
}

// the address of the C descriptor (for the calls that take it through ctypes); valid as long as the view is
PyObject * view_descriptor(View * v, PyObject *) {
    return view_resolve(v) ? PyLong_FromVoidPtr(&v->t) : nullptr;
}

PyMethodDef view_methods[] = {
    {"view", (PyCFunction)(void *)view_view, METH_FASTCALL | METH_KEYWORDS,
     "view(ne, nb, offset=0, type_=None): ggml_view_{1,2,3,4}d: same buffer, new extents/strides, offset relative to this view"},
    {"span", (PyCFunction)view_span, METH_NOARGS, "bytes from the view's first to one past its last byte"},
    {"data_ptr", (PyCFunction)view_data_ptr, METH_NOARGS, "the address of the view's first element"},
    {"_descriptor", (PyCFunction)view_descriptor, METH_NOARGS, "address of the C descriptor"},
    {nullptr, nullptr, 0, nullptr}};

PyGetSetDef view_getset[] = {
    {"__dict__", PyObject_GenericGetDict, PyObject_GenericSetDict, nullptr, nullptr},
    {nullptr, nullptr, nullptr, nullptr, nullptr}};

PyTypeObject ViewType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// ---- the calls ------------------------------------------------------------------------------------------------------

// an operand of a call: a View whose buffer exists
View * operand(PyObject * o, bool optional, bool * ok) {
    if (o == Py_None && optional) return nullptr;
    if (!PyObject_TypeCheck(o, &ViewType)) {
        PyErr_Format(PyExc_TypeError, "a Tensor is needed, not %.80s", Py_TYPE(o)->tp_name);
        *ok = false;
        return nullptr;
    }
    View * v = (View *)o;
    if (!view_resolve(v)) {
        *ok = false;
    } else if (v->device == NO_BUFFER) {
        PyErr_SetString(PyExc_AttributeError, "the tensor has no buffer: it is good for planning only");
        *ok = false;
    }
    return v;
}

const mi355x_tensor * desc(const View * v) { return v ? &v->t : nullptr; }

// the handle of `stream`, or of torch's current stream on the device
bool stream_of(PyObject * stream, int device, void ** out) {
    int64_t h = 0;
    bool    ok;
    if (stream != Py_None) {
        PyObject * s = PyObject_GetAttr(stream, s_cuda_stream);
        ok = s && to_i64(s, &h);
        Py_XDECREF(s);
    } else {
        PyObject * d = PyLong_FromLong(device);
        PyObject * s = d ? PyObject_CallOneArg(g_raw_stream, d) : nullptr;
        Py_XDECREF(d);
        ok = s && to_i64(s, &h);
        Py_XDECREF(s);
    }
    *out = (void *)(uintptr_t)h;
    return ok;
}

// run `call(stream)` with `device` current (it almost always is) and without the interpreter lock
template <typename F>
PyObject * launch(int device, PyObject * stream, F call) {
    if (!g_lib.cpy) {
        PyErr_SetString(PyExc_RuntimeError, "the library is not loaded");
        return nullptr;
    }
    int cur = device;
    if (device >= 0 && g_lib.get_device(&cur) != 0) cur = device;
    if (device < 0 && g_lib.get_device(&cur) != 0) cur = 0;
    void * st = nullptr;
    if (!stream_of(stream, device >= 0 ? device : cur, &st)) return nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    if (device >= 0 && cur != device) {
        g_lib.set_device(device);
        rc = call(st);
        g_lib.set_device(cur);
    } else {
        rc = call(st);
    }
    Py_END_ALLOW_THREADS
    if (rc != MI355X_OK) {
        raise_status(rc, nullptr);
        return nullptr;
    }
    Py_RETURN_NONE;
}

bool workspace_of(PyObject * ws, void ** ptr, size_t * size) {
    *ptr  = nullptr;
    *size = 0;
    if (ws == Py_None) return true;
    int64_t p = 0, n = 0, es = 0;
    if (!call_i64(ws, s_data_ptr, &p) || !call_i64(ws, s_numel, &n) || !call_i64(ws, s_element_size, &es)) return false;
    *ptr  = (void *)(uintptr_t)p;
    *size = (size_t)(n * es);
    return true;
}

bool real_arg(PyObject * o, float * out) {
    const double d = PyFloat_AsDouble(o);
    if (d == -1.0 && PyErr_Occurred()) return false;
    *out = (float)d;
    return true;
}
bool int_arg(PyObject * o, int32_t * out) {
    int64_t x = 0;
    if (!to_i64(o, &x)) return false;
    *out = (int32_t)x;
    return true;
}

#define NEED(k)                                                                        \
    if (n != (k)) {                                                                    \
        PyErr_Format(PyExc_TypeError, "%d arguments are needed, not %zd", (k), n);      \
        return nullptr;                                                                \
    }

// (q, k, v, mask, out, scale, max_bias, logit_softcap, prec, kernel, n_splits, workspace, stream, q_quant, tile_variant, no_alloc)
PyObject * py_flash_attn_ext(PyObject *, PyObject * const * a, Py_ssize_t n) {
    NEED(16)
    bool ok = true;
    View * q = operand(a[0], false, &ok);
    View * k = ok ? operand(a[1], false, &ok) : nullptr;
    View * v = ok ? operand(a[2], false, &ok) : nullptr;
    View * m = ok ? operand(a[3], true, &ok) : nullptr;
    View * o = ok ? operand(a[4], false, &ok) : nullptr;
    mi355x_fattn_params p;
    memset(&p, 0, sizeof(p));
    if (!ok || !real_arg(a[5], &p.scale) || !real_arg(a[6], &p.max_bias) || !real_arg(a[7], &p.logit_softcap) || !int_arg(a[8], &p.prec) ||
        !int_arg(a[9], &p.kernel) || !int_arg(a[10], &p.n_splits) || !workspace_of(a[11], &p.workspace, &p.workspace_size) ||
        !int_arg(a[13], &p.q_quant) || !int_arg(a[14], &p.tile_variant))
        return nullptr;
    const int no_alloc = PyObject_IsTrue(a[15]);
    if (no_alloc < 0) return nullptr;
    const attn_fn fn = no_alloc ? g_lib.flash_attn_ext_noalloc : g_lib.flash_attn_ext;
    return launch(q->device, a[12], [&](void * st) { return fn(&q->t, &k->t, &v->t, desc(m), &o->t, &p, st); });
}

// (src, dst, stream)
PyObject * py_cpy(PyObject *, PyObject * const * a, Py_ssize_t n) {
    NEED(3)
    bool ok = true;
    View * s = operand(a[0], false, &ok);
    View * d = ok ? operand(a[1], false, &ok) : nullptr;
    if (!ok) return nullptr;
    return launch(d->device, a[2], [&](void * st) { return g_lib.cpy(&s->t, &d->t, st); });
}

// (dst, src, idx, stream); idx: an int64 or int32 device tensor of up to three dimensions
PyObject * py_set_rows(PyObject *, PyObject * const * a, Py_ssize_t n) {
    NEED(4)
    bool ok = true;
    View * d = operand(a[0], false, &ok);
    View * s = ok ? operand(a[1], false, &ok) : nullptr;
    if (!ok) return nullptr;
    PyObject * dt = PyObject_GetAttr(a[2], s_dtype);
    if (!dt) return nullptr;
    Py_DECREF(dt);
    int64_t contiguous = 0, p = 0, dims[4] = {1, 1, 1, 1};
    if (!call_i64(a[2], s_is_contiguous, &contiguous)) return nullptr;
    if ((dt != g_int64 && dt != g_int32) || !contiguous) {
        PyErr_SetString(PyExc_AssertionError, "row indices are a contiguous int64 or int32 tensor");
        return nullptr;
    }
    PyObject * shape = PyObject_GetAttr(a[2], s_shape);
    if (!shape) return nullptr;
    const int nd = ints_of(shape, dims);
    Py_DECREF(shape);
    if (nd < 0 || !call_i64(a[2], s_data_ptr, &p)) return nullptr;
    if (nd > 3) {
        PyErr_SetString(PyExc_ValueError, "row indices have at most 3 dimensions");
        return nullptr;
    }
    int64_t ine[3] = {1, 1, 1};
    for (int i = 0; i < nd; i++) ine[nd - 1 - i] = dims[i];
    const size_t es = dt == g_int64 ? 8 : 4;
    const size_t inb[3] = {es, es * (size_t)ine[0], es * (size_t)ine[0] * (size_t)ine[1]};
    const int    bits = dt == g_int64 ? 64 : 32;
    return launch(d->device, a[3], [&](void * st) { return g_lib.set_rows(&s->t, (const void *)(uintptr_t)p, bits, ine, inb, &d->t, st); });
}

// (q_v, r, add, out, scale, workspace, stream)
PyObject * py_relpos_bias(PyObject *, PyObject * const * a, Py_ssize_t n) {
    NEED(7)
    bool ok = true;
    View * qv = operand(a[0], false, &ok);
    View * r  = ok ? operand(a[1], false, &ok) : nullptr;
    View * ad = ok ? operand(a[2], true, &ok) : nullptr;
    View * o  = ok ? operand(a[3], false, &ok) : nullptr;
    float  scale = 0.0f;
    void * ws = nullptr;
    size_t wn = 0;
    if (!ok || !real_arg(a[4], &scale) || !workspace_of(a[5], &ws, &wn)) return nullptr;
    return launch(qv->device, a[6], [&](void * st) { return g_lib.relpos_bias(&qv->t, &r->t, desc(ad), &o->t, scale, ws, wn, st); });
}

// (q_u, q_v, k, v, r, add, out, scale, kernel, n_splits, workspace, stream)
PyObject * py_flash_attn_relpos(PyObject *, PyObject * const * a, Py_ssize_t n) {
    NEED(12)
    bool ok = true;
    View * qu = operand(a[0], false, &ok);
    View * qv = ok ? operand(a[1], false, &ok) : nullptr;
    View * k  = ok ? operand(a[2], false, &ok) : nullptr;
    View * v  = ok ? operand(a[3], false, &ok) : nullptr;
    View * r  = ok ? operand(a[4], false, &ok) : nullptr;
    View * ad = ok ? operand(a[5], true, &ok) : nullptr;
    View * o  = ok ? operand(a[6], false, &ok) : nullptr;
    mi355x_fattn_params p;
    memset(&p, 0, sizeof(p));
    if (!ok || !real_arg(a[7], &p.scale) || !int_arg(a[8], &p.kernel) || !int_arg(a[9], &p.n_splits) ||
        !workspace_of(a[10], &p.workspace, &p.workspace_size))
        return nullptr;
    return launch(qu->device, a[11], [&](void * st) { return g_lib.flash_attn_relpos(&qu->t, &qv->t, &k->t, &v->t, &r->t, desc(ad), &o->t, &p, st); });
}

// bind(addresses: dict of entry point name -> address, failed, raw_stream): the loaded library
PyObject * py_bind(PyObject *, PyObject * args) {
    PyObject * d, * failed, * raw;
    if (!PyArg_ParseTuple(args, "O!OO", &PyDict_Type, &d, &failed, &raw)) return nullptr;
    Bound b;
    struct { const char * name; void * at; } want[] = {
        {"mi355x_flash_attn_ext", &b.flash_attn_ext}, {"mi355x_flash_attn_ext_noalloc", &b.flash_attn_ext_noalloc}, {"mi355x_cpy", &b.cpy},
        {"mi355x_set_rows", &b.set_rows}, {"mi355x_relpos_bias", &b.relpos_bias}, {"mi355x_flash_attn_relpos", &b.flash_attn_relpos},
        {"hipGetDevice", &b.get_device}, {"hipSetDevice", &b.set_device}};
    for (auto & w : want) {
        PyObject * x = PyDict_GetItemString(d, w.name);
        void * p = x ? PyLong_AsVoidPtr(x) : nullptr;
        if (!p) {
            if (!PyErr_Occurred()) PyErr_Format(PyExc_KeyError, "%s", w.name);
            return nullptr;
        }
        memcpy(w.at, &p, sizeof(p));
    }
    g_lib = b;
    Py_INCREF(failed);
    Py_XSETREF(g_failed, failed);
    Py_INCREF(raw);
    Py_XSETREF(g_raw_stream, raw);
    Py_RETURN_NONE;
}

// types(HostBuffer, failed, torch.uint8, torch.int32, torch.int64): what views are checked against
PyObject * py_types(PyObject *, PyObject * args) {
    PyObject * h, * failed, * u8, * i32, * i64;
    if (!PyArg_ParseTuple(args, "OOOOO", &h, &failed, &u8, &i32, &i64)) return nullptr;
    Py_INCREF(h);      Py_XSETREF(g_host_buffer, h);
    Py_INCREF(failed); Py_XSETREF(g_failed, failed);
    Py_INCREF(u8);     Py_XSETREF(g_uint8, u8);
    Py_INCREF(i32);    Py_XSETREF(g_int32, i32);
    Py_INCREF(i64);    Py_XSETREF(g_int64, i64);
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"types", py_types, METH_VARARGS, nullptr},
    {"bind", py_bind, METH_VARARGS, nullptr},
    {"flash_attn_ext", (PyCFunction)(void *)py_flash_attn_ext, METH_FASTCALL, nullptr},
    {"cpy", (PyCFunction)(void *)py_cpy, METH_FASTCALL, nullptr},
    {"set_rows", (PyCFunction)(void *)py_set_rows, METH_FASTCALL, nullptr},
    {"relpos_bias", (PyCFunction)(void *)py_relpos_bias, METH_FASTCALL, nullptr},
    {"flash_attn_relpos", (PyCFunction)(void *)py_flash_attn_relpos, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", "native host path of crispasr_amd.ggml", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) {
    ViewType.tp_name      = "crispasr_amd._host.View";
    ViewType.tp_basicsize = sizeof(View);
    ViewType.tp_flags     = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE | Py_TPFLAGS_HAVE_GC;
    ViewType.tp_dictoffset = offsetof(View, dict);
    ViewType.tp_traverse  = (traverseproc)view_traverse;
    ViewType.tp_clear     = (inquiry)view_clear;
    ViewType.tp_free      = PyObject_GC_Del;
    ViewType.tp_getattro  = PyObject_GenericGetAttr;
    ViewType.tp_setattro  = PyObject_GenericSetAttr;
    ViewType.tp_doc       = "type, ne, nb and offset over a buffer: what a ggml_tensor carries for this path";
    ViewType.tp_new       = PyType_GenericNew;
    ViewType.tp_init      = (initproc)view_init;
    ViewType.tp_dealloc   = (destructor)view_dealloc;
    ViewType.tp_methods   = view_methods;
    ViewType.tp_getset    = view_getset;
    if (PyType_Ready(&ViewType) < 0) return nullptr;
    struct { PyObject ** at; const char * name; } names[] = {
        {&s_data_ptr, "data_ptr"}, {&s_numel, "numel"}, {&s_get_device, "get_device"}, {&s_device, "device"}, {&s_index, "index"},
        {&s_dtype, "dtype"}, {&s_dim, "dim"}, {&s_is_contiguous, "is_contiguous"}, {&s_cuda_stream, "cuda_stream"}, {&s_shape, "shape"},
        {&s_element_size, "element_size"}, {&s_buf, "buf"}, {&s_type, "type"}, {&s_ne, "ne"}, {&s_nb, "nb"}, {&s_offset, "offset"}};
    for (auto & x : names)
        if (!(*x.at = PyUnicode_InternFromString(x.name))) return nullptr;
    PyObject * m = PyModule_Create(&module);
    if (!m) return nullptr;
    Py_INCREF(&ViewType);
    if (PyModule_AddObject(m, "View", (PyObject *)&ViewType) < 0) {
        Py_DECREF(&ViewType);
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
