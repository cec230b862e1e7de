// The way from Python to the kernel library's entry points, as a CPython module: what runs on the host for every operand and every launch of a
// step.  A step of few rows is bound by it: 149 launches of a prompt of 37 tokens (Gemma-2B sizes) took 13.8 us each, of which the runtime's own
// launch is 2.8.  ctypes takes 1.7 us for 17 arguments where an `Entry` takes 0.3; the look at an operand (type, layout, shape) 0.34 us in
// Python and 0.1 here, its address 0.2 and 0.08.  That prompt 1.90 to 1.54 ms (what the GPU is busy), a Tokuvik prompt of 37 tokens 4.16 to 3.24.
//
//   Entry(address, codes)   calls the function at an address: a letter of `codes` an argument (p pointer: an integer, None or a ctypes
//                           pointer; i 32-bit integer, l 64-bit integer, f float), an int as the result; the interpreter's lock is released meanwhile
//   address(t)              a tensor's address, None for None
//   make_on_gpu(error)      a function that raises `error` unless each of its arguments is None or a tensor on a GPU
//   make_dense(slow)        a function (t, name, dtype, shape=None) that returns where t is a contiguous tensor of that type (or of one of a
//                           tuple of types) and shape, and else leaves the answer to `slow`, which it hands its arguments
#include <Python.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>
#include <cstring>

#if !defined(__x86_64__) || !defined(__linux__)
#error "the calling convention below is that of x86-64 Linux"
#endif

namespace {

constexpr int kMostArguments = 48, kMostWhole = 40, kMostFloats = 8;

struct Entry {
    PyObject_HEAD
    vectorcallfunc call;
    void* function;
    int count;
    char codes[kMostArguments];
};

// By the convention of x86-64 System V, integers and pointers take their registers, then stack slots of 8 bytes, in their own order, and up to
// eight floats theirs, wherever they stand among the others; what the caller passes beyond a function's arguments is not looked at.  So one
// shape of call serves every entry point.
using Anything = int (*)(int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t,
                         int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t,
                         int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t,
                         int64_t, float, float, float, float, float, float, float, float);

bool pointer_of(PyObject* o, int64_t& to) {
    if (o == Py_None) {
        to = 0;
        return true;
    }
    if (PyLong_Check(o)) {
        to = static_cast<int64_t>(PyLong_AsUnsignedLongLong(o));
        return !PyErr_Occurred();
    }
    PyObject* value = PyObject_GetAttrString(o, "value");           // a ctypes pointer
    if (value == nullptr) {
        PyErr_Format(PyExc_TypeError, "a pointer argument is an integer, None or a ctypes pointer, not %s", Py_TYPE(o)->tp_name);
        return false;
    }
    const bool ok = value == Py_None || PyLong_Check(value);
    to = !ok || value == Py_None ? 0 : static_cast<int64_t>(PyLong_AsUnsignedLongLong(value));
    if (!ok) PyErr_Format(PyExc_TypeError, "a pointer argument is an integer, None or a ctypes pointer, not %s", Py_TYPE(o)->tp_name);
    Py_DECREF(value);
    return ok && !PyErr_Occurred();
}

PyObject* entry_call(PyObject* self, PyObject* const* args, size_t nargsf, PyObject* names) {
    const Entry* e = reinterpret_cast<Entry*>(self);
    const Py_ssize_t n = PyVectorcall_NARGS(nargsf);
    if (n != e->count || (names != nullptr && PyTuple_GET_SIZE(names) != 0)) {
        PyErr_Format(PyExc_TypeError, "this entry point takes %d arguments, got %zd", e->count, n);
        return nullptr;
    }
    int64_t w[kMostWhole] = {0};
    float f[kMostFloats] = {0.f};
    int whole = 0, floats = 0;
    for (int a = 0; a < e->count; ++a) {
        switch (e->codes[a]) {
            case 'p':
                if (!pointer_of(args[a], w[whole++])) return nullptr;
                break;
            case 'f': {
                const double v = PyFloat_AsDouble(args[a]);
                if (v == -1.0 && PyErr_Occurred()) return nullptr;
                f[floats++] = static_cast<float>(v);
                break;
            }
            default: {
                const long long v = PyLong_AsLongLong(args[a]);
                if (v == -1 && PyErr_Occurred()) return nullptr;
                if (e->codes[a] == 'i' && v != static_cast<int32_t>(v)) {
                    PyErr_Format(PyExc_OverflowError, "argument %d of an entry point does not fit 32 bits: %lld", a, v);
                    return nullptr;
                }
                w[whole++] = v;
            }
        }
    }
    int result;
    Py_BEGIN_ALLOW_THREADS
    result = reinterpret_cast<Anything>(e->function)(
        w[0], w[1], w[2], w[3], w[4], w[5], w[6], w[7], w[8], w[9], w[10], w[11], w[12], w[13], w[14], w[15], w[16], w[17], w[18], w[19],
        w[20], w[21], w[22], w[23], w[24], w[25], w[26], w[27], w[28], w[29], w[30], w[31], w[32], w[33], w[34], w[35], w[36], w[37], w[38],
        w[39], f[0], f[1], f[2], f[3], f[4], f[5], f[6], f[7]);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(result);
}

PyObject* entry_new(PyTypeObject* type, PyObject* args, PyObject* kwargs) {
    unsigned long long function;
    const char* codes;
    if ((kwargs && PyDict_Size(kwargs)) || !PyArg_ParseTuple(args, "Ks", &function, &codes)) {
        if (!PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, "Entry(address, codes)");
        return nullptr;
    }
    int whole = 0, floats = 0;
    const size_t count = std::strlen(codes);
    for (size_t a = 0; a < count; ++a) {
        if (std::strchr("pilf", codes[a]) == nullptr) {
            PyErr_SetString(PyExc_ValueError, "Entry: an argument is one of p, i, l and f");
            return nullptr;
        }
        ++(codes[a] == 'f' ? floats : whole);
    }
    if (function == 0 || count > kMostArguments || whole > kMostWhole || floats > kMostFloats) {
        PyErr_SetString(PyExc_ValueError, "Entry: no function, or more arguments than a call has room for");
        return nullptr;
    }
    Entry* e = reinterpret_cast<Entry*>(type->tp_alloc(type, 0));
    if (e == nullptr) return nullptr;
    e->call = entry_call;
    e->function = reinterpret_cast<void*>(function);
    e->count = static_cast<int>(count);
    std::memcpy(e->codes, codes, count);
    return reinterpret_cast<PyObject*>(e);
}

// A function of the module with one Python object of its own (the error to raise, or the function to ask).
struct Bound {
    PyObject_HEAD
    vectorcallfunc call;
    PyObject* own;
};

// (what torch throws is a Python error here, and no more)
template <typename F>
bool guarded(F f) {
    try {
        return f();
    } catch (const std::exception& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
    } catch (...) {
        PyErr_SetString(PyExc_RuntimeError, "an operand could not be looked at");
    }
    return false;
}

PyObject* on_gpu_call(PyObject* self, PyObject* const* args, size_t nargsf, PyObject* names) {
    const Py_ssize_t n = PyVectorcall_NARGS(nargsf);
    if (names != nullptr && PyTuple_GET_SIZE(names) != 0) {
        PyErr_SetString(PyExc_TypeError, "on_gpu takes no names");
        return nullptr;
    }
    for (Py_ssize_t a = 0; a < n; ++a) {
        if (args[a] == Py_None) continue;
        bool there = false;
        if (!THPVariable_Check(args[a])) {
            PyErr_Format(PyExc_TypeError, "a kernel operand is a tensor, not %s", Py_TYPE(args[a])->tp_name);
            return nullptr;
        }
        if (!guarded([&] {
                there = THPVariable_Unpack(args[a]).is_cuda();
                return true;
            }))
            return nullptr;
        if (!there) {
            PyErr_SetString(reinterpret_cast<Bound*>(self)->own, "a kernel operand is not on the GPU");
            return nullptr;
        }
    }
    Py_RETURN_NONE;
}

bool is_of(const at::Tensor& t, PyObject* dtype) {
    return THPDtype_Check(dtype) && reinterpret_cast<THPDtype*>(dtype)->scalar_type == t.scalar_type();
}

// Whether the common answer is yes; false also for whatever is unusual.
bool plainly_dense(PyObject* const* args, Py_ssize_t n) {
    if (n < 3 || n > 4 || !THPVariable_Check(args[0])) return false;
    const at::Tensor& t = THPVariable_Unpack(args[0]);
    bool type = is_of(t, args[2]);
    if (!type && PyTuple_CheckExact(args[2]))
        for (Py_ssize_t d = 0; d < PyTuple_GET_SIZE(args[2]) && !type; ++d) type = is_of(t, PyTuple_GET_ITEM(args[2], d));
    if (!type || t.layout() != at::kStrided || !t.is_contiguous()) return false;
    if (n == 3 || args[3] == Py_None) return true;
    if (!PyTuple_Check(args[3]) || PyTuple_GET_SIZE(args[3]) != t.dim()) return false;
    const auto sizes = t.sizes();
    for (Py_ssize_t d = 0; d < t.dim(); ++d) {
        PyObject* size = PyTuple_GET_ITEM(args[3], d);
        if (!PyLong_Check(size)) return false;
        int overflow = 0;
        if (PyLong_AsLongLongAndOverflow(size, &overflow) != sizes[d] || overflow) return false;
    }
    return true;
}

PyObject* dense_call(PyObject* self, PyObject* const* args, size_t nargsf, PyObject* names) {
    const Py_ssize_t n = PyVectorcall_NARGS(nargsf);
    if (names == nullptr || PyTuple_GET_SIZE(names) == 0) {
        const bool yes = guarded([&] { return plainly_dense(args, n); });
        if (yes) Py_RETURN_NONE;
        PyErr_Clear();
    }
    return PyObject_Vectorcall(reinterpret_cast<Bound*>(self)->own, args, nargsf & ~PY_VECTORCALL_ARGUMENTS_OFFSET, names);
}

void bound_free(PyObject* self) {
    Py_XDECREF(reinterpret_cast<Bound*>(self)->own);
    Py_TYPE(self)->tp_free(self);
}

PyTypeObject entry_type = {PyVarObject_HEAD_INIT(nullptr, 0)};
PyTypeObject bound_type = {PyVarObject_HEAD_INIT(nullptr, 0)};

PyObject* make_bound(PyObject* own, vectorcallfunc call) {
    Bound* b = reinterpret_cast<Bound*>(bound_type.tp_alloc(&bound_type, 0));
    if (b == nullptr) return nullptr;
    b->call = call;
    Py_INCREF(own);
    b->own = own;
    return reinterpret_cast<PyObject*>(b);
}
PyObject* make_on_gpu(PyObject*, PyObject* error) {
    if (!PyExceptionClass_Check(error)) {
        PyErr_SetString(PyExc_TypeError, "make_on_gpu takes the class of the error to raise");
        return nullptr;
    }
    return make_bound(error, on_gpu_call);
}
PyObject* make_dense(PyObject*, PyObject* slow) { return make_bound(slow, dense_call); }

PyObject* address(PyObject*, PyObject* t) {
    if (t == Py_None) Py_RETURN_NONE;
    if (!THPVariable_Check(t)) {
        PyErr_Format(PyExc_TypeError, "a tensor or None, not %s", Py_TYPE(t)->tp_name);
        return nullptr;
    }
    const void* at = nullptr;
    if (!guarded([&] {
            at = THPVariable_Unpack(t).data_ptr();
            return true;
        }))
        return nullptr;
    return PyLong_FromUnsignedLongLong(reinterpret_cast<uintptr_t>(at));
}

PyMethodDef methods[] = {{"address", address, METH_O, "A tensor's address; None for None."},
                         {"make_on_gpu", make_on_gpu, METH_O, "A function that raises the error unless every operand is on a GPU."},
                         {"make_dense", make_dense, METH_O, "A function that looks at an operand, and asks the given one where the answer is not plainly yes."},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "launch_door", "From Python to the kernel library's entry points.", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_launch_door() {
    entry_type.tp_name = "launch_door.Entry";
    entry_type.tp_basicsize = sizeof(Entry);
    entry_type.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL;
    entry_type.tp_vectorcall_offset = offsetof(Entry, call);
    entry_type.tp_call = PyVectorcall_Call;
    entry_type.tp_new = entry_new;
    bound_type.tp_name = "launch_door.Bound";
    bound_type.tp_basicsize = sizeof(Bound);
    bound_type.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL;
    bound_type.tp_vectorcall_offset = offsetof(Bound, call);
    bound_type.tp_call = PyVectorcall_Call;
    bound_type.tp_dealloc = bound_free;
    if (PyType_Ready(&entry_type) < 0 || PyType_Ready(&bound_type) < 0) return nullptr;
    PyObject* m = PyModule_Create(&module);
    if (m == nullptr) return nullptr;
    Py_INCREF(&entry_type);
    if (PyModule_AddObject(m, "Entry", reinterpret_cast<PyObject*>(&entry_type)) < 0) {
        Py_DECREF(&entry_type);
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
