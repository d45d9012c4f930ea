// The package's calls without ctypes: a CPython module that reads the handles, the scheme and the numbers of a call from the
// Python objects and calls the C ABI (include/cubek_quant.h).
//
// A call that launches one kernel takes the HIP runtime 3.2 us of the host.  Through ctypes (a lookup of the scheme's
// struct by its hash, a cached struct per handle, a conversion per argument) the package added 1.2 us to that: quantize
// and dequantize of bf16 [64, 1024] 8.9 us, host-bound.  Nothing is kept from call to call here; the structs live on the
// stack for the time of the call.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstring>
#include <initializer_list>
#include <utility>

#include "../../include/cubek_quant.h"

namespace {

PyObject *g_handle_type, *g_scheme_type;  // TensorHandleRef, QuantScheme
PyObject *s_handle, *s_shape, *s_strides, *s_elem_size, *s_as_c, *s_to_c, *s_value, *s_param, *s_store, *s_level, *s_mode, *s_block_size, *s_dims;

// A new reference that goes with the scope.
struct Ref {
    PyObject* p;
    explicit Ref(PyObject* p) : p(p) {}
    Ref(const Ref&) = delete;
    ~Ref() { Py_XDECREF(p); }
    explicit operator bool() const { return p != nullptr; }
};

// int(o), as ctypes' integer types take it: the low bits.
bool number(PyObject* o, uint64_t* out) {
    if (PyLong_Check(o)) {
        *out = PyLong_AsUnsignedLongLongMask(o);
    } else {
        const Ref n(PyNumber_Long(o));
        if (!n) return false;
        *out = PyLong_AsUnsignedLongLongMask(n.p);
    }
    return !(*out == ~0ull && PyErr_Occurred());
}

// What ctypes takes for an integer argument: an int, or a ctypes integer.
bool integer(PyObject* o, uint64_t* out) {
    if (PyLong_Check(o)) return number(o, out);
    const Ref v(PyObject_GetAttr(o, s_value));
    if (!v || !PyLong_Check(v.p)) {
        PyErr_Format(PyExc_TypeError, "an int is needed, not %s", Py_TYPE(o)->tp_name);
        return false;
    }
    return number(v.p, out);
}

// `size` bytes of a ctypes object.
bool bytes_of(PyObject* o, void* out, Py_ssize_t size) {
    Py_buffer b;
    if (PyObject_GetBuffer(o, &b, PyBUF_SIMPLE)) return false;
    const bool fits = b.len == size;
    if (fits)
        std::memcpy(out, b.buf, static_cast<size_t>(size));
    else
        PyErr_Format(PyExc_TypeError, "%s holds %zd bytes, not %zd", Py_TYPE(o)->tp_name, b.len, size);
    PyBuffer_Release(&b);
    return fits;
}

// What ctypes takes for c_void_p: an int, None, a ctypes pointer.
bool pointer(PyObject* o, void** out) {
    uint64_t n = 0;
    if (o == Py_None) {
        *out = nullptr;
    } else if (PyLong_Check(o)) {
        if (!number(o, &n)) return false;
        *out = reinterpret_cast<void*>(n);
    } else if (PyBytes_Check(o) || !PyObject_CheckBuffer(o)) {
        PyErr_Format(PyExc_TypeError, "a device pointer is an int, not %s", Py_TYPE(o)->tp_name);
        return false;
    } else {
        return bytes_of(o, out, sizeof(void*));
    }
    return true;
}

// A tensor argument: the struct and what keeps its arrays for the time of the call.
struct Tensor {
    cq_tensor t{};
    uint64_t dims[2 * CQ_MAX_RANK];
    PyObject* keep = nullptr;
    ~Tensor() { Py_XDECREF(keep); }

    // `take`: number for what a handle holds, integer for an argument
    static bool extents(PyObject* o, uint64_t* out, Py_ssize_t* n, bool (*take)(PyObject*, uint64_t*)) {
        const Ref fast(PySequence_Fast(o, "shape and strides are sequences"));
        if (!fast) return false;
        *n = PySequence_Fast_GET_SIZE(fast.p);
        for (Py_ssize_t i = 0; i < *n && i < CQ_MAX_RANK; i++)
            if (!take(PySequence_Fast_GET_ITEM(fast.p, i), out + i)) return false;
        return true;
    }

    // A TensorHandleRef is read here; anything else that stands for one gives its cq_tensor.
    bool read(PyObject* o) {
        if (reinterpret_cast<PyObject*>(Py_TYPE(o)) != g_handle_type) {
            keep = PyObject_CallMethodNoArgs(o, s_as_c);
            return keep && bytes_of(keep, &t, sizeof(t));
        }
        const Ref handle(PyObject_GetAttr(o, s_handle)), size(PyObject_GetAttr(o, s_elem_size));
        const Ref shape(PyObject_GetAttr(o, s_shape)), strides(PyObject_GetAttr(o, s_strides));
        uint64_t elem_size = 0;
        Py_ssize_t rank = 0, ranks = 0;
        if (!handle || !size || !shape || !strides || !pointer(handle.p, &t.ptr) || !integer(size.p, &elem_size) ||
            !extents(shape.p, dims, &rank, number) || !extents(strides.p, dims + CQ_MAX_RANK, &ranks, number))
            return false;
        if (ranks != rank) {
            if (ranks > rank) {
                PyErr_SetString(PyExc_IndexError, "more strides than extents");
                return false;
            }
            for (Py_ssize_t i = ranks; i < rank && i < CQ_MAX_RANK; i++) dims[CQ_MAX_RANK + i] = 0;
        }
        t.shape = dims;
        t.strides = dims + CQ_MAX_RANK;
        t.rank = static_cast<uint32_t>(rank);  // above CQ_MAX_RANK: refused before an extent is read
        t.elem_size = static_cast<uint32_t>(elem_size);
        return true;
    }
};

bool read_scheme(PyObject* o, cq_scheme* s) {
    std::memset(s, 0, sizeof(*s));
    if (reinterpret_cast<PyObject*>(Py_TYPE(o)) != g_scheme_type) {
        const Ref c(PyObject_CallMethodNoArgs(o, s_to_c));
        return c && bytes_of(c.p, s, sizeof(*s));
    }
    const auto field = [o](PyObject* name, uint8_t* out) {
        const Ref v(PyObject_GetAttr(o, name));
        uint64_t n = 0;
        if (!v || !number(v.p, &n)) return false;
        *out = static_cast<uint8_t>(n);
        return true;
    };
    if (!field(s_value, &s->value) || !field(s_param, &s->param) || !field(s_store, &s->store) || !field(s_mode, &s->mode)) return false;
    const Ref level(PyObject_GetAttr(o, s_level));
    if (!level) return false;
    const Ref block(PyObject_GetAttr(level.p, s_block_size));
    if (!block) return false;
    s->level = CQ_LEVEL_TENSOR;
    if (block.p == Py_None) return true;
    s->level = CQ_LEVEL_BLOCK;
    const Ref dims(PyObject_GetAttr(block.p, s_dims));
    if (!dims) return false;
    const Ref fast(PySequence_Fast(dims.p, "block extents are a sequence"));
    if (!fast) return false;
    const Py_ssize_t n = PySequence_Fast_GET_SIZE(fast.p);
    if (n > CQ_MAX_BLOCK_DIMS) {
        PyErr_SetString(PyExc_IndexError, "too many block extents");
        return false;
    }
    s->block_rank = static_cast<uint8_t>(n);
    for (Py_ssize_t i = 0; i < n; i++) {
        uint64_t v = 0;
        if (!number(PySequence_Fast_GET_ITEM(fast.p, i), &v)) return false;
        s->block[i] = static_cast<uint8_t>(v);
    }
    return true;
}

bool count(Py_ssize_t got, Py_ssize_t want) {
    if (got != want) PyErr_Format(PyExc_TypeError, "%zd arguments, not %zd", got, want);
    return got == want;
}

// The status of a call, made without the interpreter's lock (a launch waits while its queue is full).
template <class Call>
PyObject* status_of(Call call) {
    cq_status st;
    Py_BEGIN_ALLOW_THREADS
    st = call();
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(st);
}

// Arguments: stream, `kTensors` tensors, scheme, element type; the caller reads what comes after them.
template <int kTensors>
struct Common {
    void* stream;
    Tensor t[kTensors];
    cq_scheme scheme;
    cq_dtype elem;
    static constexpr Py_ssize_t kArgs = kTensors + 3;

    bool read(PyObject* const* a) {
        if (!pointer(a[0], &stream)) return false;
        for (int i = 0; i < kTensors; i++)
            if (!t[i].read(a[1 + i])) return false;
        return read_scheme(a[1 + kTensors], &scheme) && read_elem(a[2 + kTensors], &elem);
    }
    static bool read_elem(PyObject* o, cq_dtype* out) {
        uint64_t n = 0;
        if (!number(o, &n)) return false;
        *out = static_cast<cq_dtype>(static_cast<int>(n));
        return true;
    }
    cq_stream_t s() const { return static_cast<cq_stream_t>(stream); }
};

PyObject* quantize(PyObject*, PyObject* const* a, Py_ssize_t n) {
    Common<4> c;
    if (!count(n, c.kArgs) || !c.read(a)) return nullptr;
    return status_of([&] { return cq_quantize(c.s(), &c.t[0].t, &c.t[1].t, &c.t[2].t, &c.t[3].t, &c.scheme, c.elem); });
}

PyObject* dequantize(PyObject*, PyObject* const* a, Py_ssize_t n) {
    Common<3> c;
    if (!count(n, c.kArgs) || !c.read(a)) return nullptr;
    return status_of([&] { return cq_dequantize(c.s(), &c.t[0].t, &c.t[1].t, &c.t[2].t, &c.scheme, c.elem); });
}

PyObject* compute_scales(PyObject*, PyObject* const* a, Py_ssize_t n) {
    Common<2> c;
    void* workspace;
    uint64_t bytes;
    if (!count(n, c.kArgs + 2) || !c.read(a) || !pointer(a[5], &workspace) || !integer(a[6], &bytes)) return nullptr;
    return status_of([&] { return cq_compute_scales(c.s(), &c.t[0].t, &c.t[1].t, &c.scheme, c.elem, workspace, bytes); });
}

PyObject* quantize_dynamic(PyObject*, PyObject* const* a, Py_ssize_t n) {
    Common<3> c;
    void* workspace;
    uint64_t bytes;
    if (!count(n, c.kArgs + 2) || !c.read(a) || !pointer(a[6], &workspace) || !integer(a[7], &bytes)) return nullptr;
    return status_of([&] { return cq_quantize_dynamic(c.s(), &c.t[0].t, &c.t[1].t, &c.t[2].t, &c.scheme, c.elem, workspace, bytes); });
}

PyObject* quantize_dynamic_static(PyObject*, PyObject* const* a, Py_ssize_t n) {
    Common<3> c;
    if (!count(n, c.kArgs) || !c.read(a)) return nullptr;
    return status_of([&] { return cq_quantize_dynamic_static(c.s(), &c.t[0].t, &c.t[1].t, &c.t[2].t, &c.scheme, c.elem); });
}

// stream, values, params, scheme, x, y, elem, y_elem
PyObject* gemv(PyObject*, PyObject* const* a, Py_ssize_t n) {
    void* stream;
    Tensor values, params, x, y;
    cq_scheme scheme;
    cq_dtype elem, y_elem;
    if (!count(n, 8) || !pointer(a[0], &stream) || !values.read(a[1]) || !params.read(a[2]) || !read_scheme(a[3], &scheme) || !x.read(a[4]) ||
        !y.read(a[5]) || !Common<1>::read_elem(a[6], &elem) || !Common<1>::read_elem(a[7], &y_elem))
        return nullptr;
    return status_of([&] { return cq_gemv_quantized(static_cast<cq_stream_t>(stream), &values.t, &params.t, &scheme, &x.t, &y.t, elem, y_elem); });
}

// stream, input, output, axis, elem, workspace, bytes
PyObject* max_abs(PyObject*, PyObject* const* a, Py_ssize_t n) {
    void *stream, *workspace;
    Tensor in, out;
    uint64_t axis, bytes;
    cq_dtype elem;
    if (!count(n, 7) || !pointer(a[0], &stream) || !in.read(a[1]) || !out.read(a[2]) || !integer(a[3], &axis) || !Common<1>::read_elem(a[4], &elem) ||
        !pointer(a[5], &workspace) || !integer(a[6], &bytes))
        return nullptr;
    return status_of([&] { return cq_reduce_max_abs(static_cast<cq_stream_t>(stream), &in.t, &out.t, static_cast<uint32_t>(axis), elem, workspace, bytes); });
}

// stream, input, output, shape, packing
PyObject* repack(PyObject*, PyObject* const* a, Py_ssize_t n) {
    void* stream;
    Tensor in, out;
    uint64_t shape[CQ_MAX_RANK], packing;
    Py_ssize_t rank;
    if (!count(n, 5) || !pointer(a[0], &stream) || !in.read(a[1]) || !out.read(a[2]) || !Tensor::extents(a[3], shape, &rank, integer) || !integer(a[4], &packing))
        return nullptr;
    return status_of([&] {
        return cq_into_contiguous_packed(static_cast<cq_stream_t>(stream), &in.t, &out.t, shape, static_cast<uint32_t>(rank), static_cast<uint32_t>(packing));
    });
}

template <class F>
constexpr PyMethodDef method(const char* name, F f) {
    return {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)), METH_FASTCALL, nullptr};
}

PyObject* bind(PyObject*, PyObject* args) {
    PyObject *handle, *scheme;
    if (!PyArg_ParseTuple(args, "OO", &handle, &scheme)) return nullptr;
    Py_INCREF(handle);
    Py_INCREF(scheme);
    Py_XSETREF(g_handle_type, handle);
    Py_XSETREF(g_scheme_type, scheme);
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    method("quantize", quantize), method("dequantize", dequantize), method("compute_scales", compute_scales),
    method("quantize_dynamic", quantize_dynamic), method("quantize_dynamic_static", quantize_dynamic_static),
    method("gemv", gemv), method("max_abs", max_abs), method("repack", repack),
    {"bind", bind, METH_VARARGS, "bind(TensorHandleRef, QuantScheme)"}, {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_call", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__call() {
    const std::initializer_list<std::pair<PyObject**, const char*>> names = {
        {&s_handle, "handle"}, {&s_shape, "shape"}, {&s_strides, "strides"}, {&s_elem_size, "elem_size"}, {&s_as_c, "as_c"},
        {&s_to_c, "to_c"}, {&s_value, "value"}, {&s_param, "param"}, {&s_store, "store"}, {&s_level, "level"},
        {&s_mode, "mode"}, {&s_block_size, "block_size"}, {&s_dims, "dims"},
    };
    for (const auto& [at, name] : names)
        if (!(*at = PyUnicode_InternFromString(name))) return nullptr;
    return PyModule_Create(&module);
}
