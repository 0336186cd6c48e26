// The per-layer entry points of a decode step, called straight from torch
// tensors. Through ctypes a fused append + attend spends about half of its 11.4
// us on the host in Python: four descriptors keyed by (pointer, type, shape,
// strides), a slot tuple, two foreign calls with nine converted arguments. Read
// from the tensors here, the call takes 7.7 us (30-layer frame of one stream),
// less than its two short launches do on the GPU.
//
// Every function returns the runtime's code (0 or negative), or 1 where an
// argument is not in the plain form it reads: an exact torch.Tensor on the GPU
// (contiguous where the Python wrapper would have made it so), exact ints in
// lists or tuples. Nothing has happened then, and the caller takes its general
// path, which converts or refuses the call; a stream that cannot be bound goes
// there too. Nothing is kept between calls.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <climits>

#include <torch/csrc/autograd/python_variable.h>

#include "kvrt.h"

namespace {

constexpr int kMaxSlots = 64, kMaxPositions = 256;
constexpr long kGeneral = 1;

struct Api {
    decltype(&kvrt_bind_stream) bind;
    decltype(&kvrt_append_attend_async) append_attend;
    decltype(&kvrt_attend_decode_async) attend;
    decltype(&kvrt_attend_talker_async) talker;
    decltype(&kvrt_write_positions_async) write;
    decltype(&kvrt_append_gather_async) gather;
    decltype(&kvrt_attend_tensors_async) tensors;
} api;

PyObject *talker_mask_type;

bool read_int(PyObject *o, int32_t &out) {
    if (!PyLong_CheckExact(o)) return false;
    int over = 0;
    const long v = PyLong_AsLongAndOverflow(o, &over);
    if (over || v < INT_MIN || v > INT_MAX) return false;
    out = (int32_t)v;
    return true;
}

bool read_float(PyObject *o, float &out) {
    if (!PyFloat_CheckExact(o)) return false;
    out = (float)PyFloat_AS_DOUBLE(o);
    return true;
}

// Items of an exact list or tuple (borrowed), or -1.
Py_ssize_t items(PyObject *o, PyObject **&at) {
    if (!PyList_CheckExact(o) && !PyTuple_CheckExact(o)) return -1;
    at = PySequence_Fast_ITEMS(o);
    return PySequence_Fast_GET_SIZE(o);
}

int read_ints(PyObject *o, int32_t *out, int cap) {
    PyObject **at;
    const Py_ssize_t n = items(o, at);
    if (n < 0 || n > cap) return -1;
    for (Py_ssize_t i = 0; i < n; ++i)
        if (!read_int(at[i], out[i])) return -1;
    return (int)n;
}

int dtype_code(at::ScalarType t) {
    switch (t) {
        case at::kBFloat16: return KVRT_BF16;
        case at::kChar: return KVRT_INT8;
        case at::kFloat: return KVRT_FP32;
        case at::kBool: return KVRT_BOOL;
        case at::kInt: return KVRT_INT32;
        case at::kLong: return KVRT_INT64;
        default: return -1;
    }
}

bool read_tensor(PyObject *o, bool contiguous, kvrt_tensor &d) {
    if (!THPVariable_CheckExact(o)) return false;
    const at::Tensor &t = THPVariable_Unpack(o);
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || t.dim() > KVRT_MAX_RANK) return false;
    if (contiguous && !t.is_contiguous()) return false;
    d = kvrt_tensor{};
    d.dtype = dtype_code(t.scalar_type());
    if (d.dtype < 0) return false;
    d.data = t.data_ptr();
    d.ndim = (int32_t)t.dim();
    for (int i = 0; i < d.ndim; ++i) {
        d.dims[i] = t.size(i);
        d.strides[i] = t.stride(i);
    }
    return true;
}

bool read_mask(PyObject *o, kvrt_talker_mask &m) {
    if ((PyObject *)Py_TYPE(o) != talker_mask_type) return false;
    static const char *const names[6] = {"prefix_start",   "audio_start",           "prefix_position",
                                         "audio_position", "prefix_attention_mode", "visible_prefix_count"};
    int32_t *const at[6] = {&m.prefix_start,   &m.audio_start,           &m.prefix_position,
                            &m.audio_position, &m.prefix_attention_mode, &m.visible_prefix_count};
    for (int i = 0; i < 6; ++i) {
        PyObject *v = PyObject_GetAttrString(o, names[i]);
        const bool ok = v && read_int(v, *at[i]);
        Py_XDECREF(v);
        if (!ok) return false;
    }
    PyObject *v = PyObject_GetAttrString(o, "prefix_log_gate");
    const bool ok = v && read_float(v, m.prefix_log_gate);
    Py_XDECREF(v);
    return ok;
}

// The leading arguments of a runtime call: context, stream, layer, slots.
struct Head {
    kvrt_ctx *ctx;
    void *stream;
    int32_t layer, n, slots[kMaxSlots];

    bool read(PyObject *const *a) {
        ctx = static_cast<kvrt_ctx *>(PyLong_AsVoidPtr(a[0]));
        stream = PyLong_AsVoidPtr(a[1]);
        if (!ctx || !read_int(a[2], layer)) return false;
        n = read_ints(a[3], slots, kMaxSlots);
        return n >= 0;
    }
    bool bind() const { return api.bind(ctx, stream) == KVRT_OK; }
};

// Runs body (parse, then call), any C++ or Python error of the parse meaning
// the general path.
template <class F>
PyObject *guarded(Py_ssize_t nargs, Py_ssize_t want, F body) {
    long rc = kGeneral;
    try {
        if (nargs == want) rc = body();
    } catch (...) {  // e.g. a tensor without storage
        rc = kGeneral;
    }
    if (PyErr_Occurred()) PyErr_Clear();
    return PyLong_FromLong(rc);
}

// The runtime call, the parse done. An exception out of it (its vectors can
// fail to allocate) is a device error and not the general path's to repeat: the
// call may have mapped pages or enqueued work. The interpreter lock is held
// again before anything else runs.
template <class F>
long without_gil(F call) {
    long rc;
    PyThreadState *const thread = PyEval_SaveThread();
    try {
        rc = call();
    } catch (...) {
        rc = KVRT_EDEVICE;
    }
    PyEval_RestoreThread(thread);
    return rc;
}

// (ctx, stream, layer, slots, scale, q, k, v, out)
PyObject *append_attend(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    return guarded(nargs, 9, [&]() -> long {
        Head h;
        float scale;
        kvrt_tensor q, k, v, o;
        if (!h.read(a) || !read_float(a[4], scale) || !read_tensor(a[5], true, q) || !read_tensor(a[6], true, k) ||
            !read_tensor(a[7], true, v) || !read_tensor(a[8], false, o) || !h.bind())
            return kGeneral;
        return without_gil([&] { return api.append_attend(h.ctx, h.layer, h.n, h.slots, &q, &k, &v, &o, scale); });
    });
}

// (ctx, stream, layer, slots, scale, q, out)
PyObject *attend(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    return guarded(nargs, 7, [&]() -> long {
        Head h;
        float scale;
        kvrt_tensor q, o;
        if (!h.read(a) || !read_float(a[4], scale) || !read_tensor(a[5], true, q) || !read_tensor(a[6], false, o) ||
            !h.bind())
            return kGeneral;
        return without_gil([&] { return api.attend(h.ctx, h.layer, h.n, h.slots, &q, &o, scale); });
    });
}

// (ctx, stream, layer, slots, scale, q, out, masks)
PyObject *attend_talker(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    return guarded(nargs, 8, [&]() -> long {
        Head h;
        float scale;
        kvrt_tensor q, o;
        kvrt_talker_mask m[kMaxSlots];
        PyObject **at = nullptr;
        if (!h.read(a) || !read_float(a[4], scale) || !read_tensor(a[5], true, q) || !read_tensor(a[6], false, o) ||
            items(a[7], at) != h.n)
            return kGeneral;
        for (int i = 0; i < h.n; ++i)
            if (!read_mask(at[i], m[i])) return kGeneral;
        if (!h.bind()) return kGeneral;
        return without_gil([&] { return api.talker(h.ctx, h.layer, h.n, h.slots, &q, &o, scale, m); });
    });
}

// (ctx, stream, layer, slots, positions, k, v)
PyObject *write_positions(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    return guarded(nargs, 7, [&]() -> long {
        Head h;
        kvrt_tensor k, v;
        int32_t pos[kMaxPositions];
        PyObject **rows;
        Py_ssize_t n_rows;
        if (!h.read(a) || (n_rows = items(a[4], rows)) < 0 || !read_tensor(a[5], false, k) ||
            !read_tensor(a[6], false, v))
            return kGeneral;
        int n = 0;
        for (Py_ssize_t i = 0; i < n_rows; ++i) {
            const int got = read_ints(rows[i], pos + n, kMaxPositions - n);
            if (got < 0) return kGeneral;
            n += got;
        }
        // other counts and empty writes are the general path's to answer
        if (k.ndim != 4 || k.dims[2] == 0 || n != k.dims[0] * k.dims[2] || !h.bind()) return kGeneral;
        return without_gil([&] { return api.write(h.ctx, h.layer, h.n, h.slots, pos, &k, &v); });
    });
}

// (ctx, stream, layer, slots, k, v, out_k, out_v, mask or None)
PyObject *append_gather(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    return guarded(nargs, 9, [&]() -> long {
        Head h;
        kvrt_tensor k, v, ok, ov, m;
        const bool masked = a[8] != Py_None;
        if (!h.read(a) || !read_tensor(a[4], false, k) || !read_tensor(a[5], false, v) ||
            !read_tensor(a[6], false, ok) || !read_tensor(a[7], false, ov) ||
            (masked && !read_tensor(a[8], false, m)) || !h.bind())
            return kGeneral;
        return without_gil([&] {
            return api.gather(h.ctx, h.layer, h.n, h.slots, &k, &v, nullptr, &ok, &ov, masked ? &m : nullptr);
        });
    });
}

// (stream, scale, window, q, k, v, lengths, out)
PyObject *attend_tensors(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    return guarded(nargs, 8, [&]() -> long {
        float scale;
        int32_t window;
        kvrt_tensor q, k, v, len, o;
        void *stream = PyLong_AsVoidPtr(a[0]);
        if (!read_float(a[1], scale) || !read_int(a[2], window) || !read_tensor(a[3], true, q) ||
            !read_tensor(a[4], false, k) || !read_tensor(a[5], false, v) || !read_tensor(a[6], true, len) ||
            len.dtype != KVRT_INT32 || !read_tensor(a[7], false, o))
            return kGeneral;
        return without_gil([&] {
            return api.tensors(&q, &k, &v, static_cast<const int32_t *>(len.data), nullptr, &o, scale, window, stream);
        });
    });
}

// (mask type, address of each Api member in order): once, after loading
PyObject *connect(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    void *p[7];
    if (nargs != 8) {
        PyErr_SetString(PyExc_TypeError, "connect takes the mask type and seven addresses");
        return nullptr;
    }
    for (int i = 0; i < 7; ++i) {
        p[i] = PyLong_AsVoidPtr(a[i + 1]);
        if (PyErr_Occurred()) return nullptr;
    }
    Py_INCREF(a[0]);
    Py_XDECREF(talker_mask_type);
    talker_mask_type = a[0];
    api.bind = reinterpret_cast<decltype(api.bind)>(p[0]);
    api.append_attend = reinterpret_cast<decltype(api.append_attend)>(p[1]);
    api.attend = reinterpret_cast<decltype(api.attend)>(p[2]);
    api.talker = reinterpret_cast<decltype(api.talker)>(p[3]);
    api.write = reinterpret_cast<decltype(api.write)>(p[4]);
    api.gather = reinterpret_cast<decltype(api.gather)>(p[5]);
    api.tensors = reinterpret_cast<decltype(api.tensors)>(p[6]);
    Py_RETURN_NONE;
}

#define KVRT_METHOD(f) {#f, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {KVRT_METHOD(append_attend),   KVRT_METHOD(attend),        KVRT_METHOD(attend_talker),
                         KVRT_METHOD(write_positions), KVRT_METHOD(append_gather), KVRT_METHOD(attend_tensors),
                         KVRT_METHOD(connect),         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "kvrt_pycall", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_kvrt_pycall() { return PyModule_Create(&module); }
