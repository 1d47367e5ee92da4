// The host path of a call: device pointers of tensors and launches of the C-ABI library without ctypes.
//
// A small kernel takes 2 to 4 us, and with ctypes a call took 6.5 to 10 us of host: about 0.7 us for the checks and the address of each
// tensor in Python, and 2 us to convert the arguments.  Both are done here, with the same checks and messages; bind() makes a function
// of every entry point that launches work, from its own declaration in spiral_mi355.h.  (us a call with the queue kept full, ctypes
// / here: a four-layer stack on packed weights 7.2 / 5.6, one on row-major weights 11.4 / 7.1, the CEM update 76 / 63, a GEMM of 16 x 16 x 296
// 7.6 / 5.4, a sampled softmax of 32 rows with its outputs allocated 11.7 / 8.7.)  What is left is the runtime's launch, about 4 us.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include <dlfcn.h>

#include <exception>
#include <memory>
#include <new>
#include <tuple>
#include <type_traits>
#include <utility>

#include "spiral_mi355.h"

namespace {

PyObject* g_calls = nullptr;      // lists of the tape being recorded: (function, arguments but the stream), tensors
PyObject* g_keep = nullptr;
PyObject* g_void_p = nullptr;     // ctypes.c_void_p
PyObject* g_byref = nullptr;      // the type of ctypes.byref(...)
PyObject* g_cdata = nullptr;      // what ctypes arrays and structures are instances of

// ---- arguments: what the caller's objects become; false with an exception set if they do not fit ----
constexpr Py_ssize_t MOST = 16;   // elements of a host array given as a list or tuple that need no allocation

bool as_integer(PyObject* o, unsigned long long& v) {      // as ctypes: the low bits of any integer
    if (PyLong_Check(o)) {
        v = PyLong_AsUnsignedLongLongMask(o);
    } else {
        PyObject* i = PyNumber_Index(o);
        if (i == nullptr) return false;
        v = PyLong_AsUnsignedLongLongMask(i);
        Py_DECREF(i);
    }
    return !(v == (unsigned long long)-1 && PyErr_Occurred());
}

bool as_address(PyObject* o, void*& p) {                   // None, an integer or a c_void_p
    if (o == Py_None) {
        p = nullptr;
        return true;
    }
    if (PyLong_Check(o)) {
        p = PyLong_AsVoidPtr(o);
        return !(p == nullptr && PyErr_Occurred());
    }
    const int is_void_p = PyObject_IsInstance(o, g_void_p);
    if (is_void_p < 0) return false;
    if (is_void_p == 0) {
        PyErr_Format(PyExc_TypeError, "an address is None, an integer or a c_void_p, not %s", Py_TYPE(o)->tp_name);
        return false;
    }
    PyObject* v = PyObject_GetAttrString(o, "value");
    if (v == nullptr) return false;
    const bool ok = as_address(v, p);
    Py_DECREF(v);
    return ok;
}

template <typename T, typename = void>
struct Arg;

template <typename T>
struct Arg<T, std::enable_if_t<std::is_integral_v<T>>> {
    T value = 0;
    bool load(PyObject* o) {
        unsigned long long v = 0;
        if (!as_integer(o, v)) return false;
        value = (T)v;
        return true;
    }
};

template <typename T>
struct Arg<T, std::enable_if_t<std::is_floating_point_v<T>>> {
    T value = 0;
    bool load(PyObject* o) {
        const double v = PyFloat_AsDouble(o);
        if (v == -1.0 && PyErr_Occurred()) return false;
        value = (T)v;
        return true;
    }
};

template <typename T>
struct Arg<T*> {
    typedef std::remove_const_t<T> Element;
    static constexpr bool HOST_ARRAY = std::is_pointer_v<Element> || std::is_same_v<T, const int32_t>;
    T* value = nullptr;
    typedef std::conditional_t<HOST_ARRAY, Element, char> Stored;
    Stored few[HOST_ARRAY ? MOST : 1];
    std::unique_ptr<Stored[]> many;
    Py_buffer buffer{};
    Arg() = default;
    Arg(const Arg&) = delete;
    ~Arg() {
        if (buffer.obj != nullptr) PyBuffer_Release(&buffer);
    }
    bool take_buffer(PyObject* o) {
        if (PyObject_GetBuffer(o, &buffer, PyBUF_SIMPLE) != 0) return false;
        value = (T*)buffer.buf;
        return true;
    }
    bool load(PyObject* o) {
        if constexpr (HOST_ARRAY) {
            if (PyTuple_Check(o) || PyList_Check(o)) {
                const Py_ssize_t n = PySequence_Fast_GET_SIZE(o);
                Stored* elements = few;
                if (n > MOST) {
                    many.reset(new (std::nothrow) Stored[n]);
                    elements = many.get();
                    if (elements == nullptr) {
                        PyErr_NoMemory();
                        return false;
                    }
                }
                for (Py_ssize_t i = 0; i < n; ++i) {
                    PyObject* e = PySequence_Fast_GET_ITEM(o, i);
                    if constexpr (std::is_pointer_v<Element>) {
                        void* p = nullptr;
                        if (!as_address(e, p)) return false;
                        elements[i] = (Element)p;
                    } else {
                        unsigned long long v = 0;
                        if (!as_integer(e, v)) return false;
                        elements[i] = (Element)v;
                    }
                }
                value = elements;
                return true;
            }
        }
        if (o == Py_None || PyLong_Check(o) || PyObject_IsInstance(o, g_void_p) == 1) {
            void* p = nullptr;
            if (!as_address(o, p)) return false;
            value = (T*)p;
            return true;
        }
        if ((PyObject*)Py_TYPE(o) == g_byref) {            // byref(x): the memory of x (no offset is given anywhere here)
            PyObject* target = PyObject_GetAttrString(o, "_obj");
            if (target == nullptr) return false;
            const bool ok = take_buffer(target);
            Py_DECREF(target);
            return ok;
        }
        const int is_cdata = PyObject_IsInstance(o, g_cdata);   // ctypes arrays and structures; no other buffer, as with ctypes
        if (is_cdata < 0) return false;
        if (is_cdata == 0) {
            PyErr_Format(PyExc_TypeError, "an address is None, an integer or an object of ctypes, not %s", Py_TYPE(o)->tp_name);
            return false;
        }
        return take_buffer(o);
    }
};

// ---- one function per entry point ----
template <int ID, typename F>
struct Entry;
template <int ID, typename... A>
struct Entry<ID, int(A...)> {
    static inline int (*fn)(A...) = nullptr;
    static inline PyObject* self = nullptr;
    static inline const char* name = nullptr;

    template <size_t... I>
    static PyObject* run(PyObject* const* given, std::index_sequence<I...>) {
        std::tuple<Arg<A>...> args;
        if (!(std::get<I>(args).load(given[I]) && ...)) return nullptr;
        int rc = 0;
        Py_BEGIN_ALLOW_THREADS
        rc = fn(std::get<I>(args).value...);
        Py_END_ALLOW_THREADS
        if (rc == 0 && g_calls != nullptr) {               // the last argument is the stream
            PyObject* kept = PyTuple_New(sizeof...(A) - 1);
            if (kept == nullptr) return nullptr;
            for (size_t i = 0; i + 1 < sizeof...(A); ++i) {
                Py_INCREF(given[i]);
                PyTuple_SET_ITEM(kept, i, given[i]);
            }
            PyObject* call = PyTuple_Pack(2, self, kept);
            Py_DECREF(kept);
            if (call == nullptr) return nullptr;
            const int failed = PyList_Append(g_calls, call);
            Py_DECREF(call);
            if (failed != 0) return nullptr;
        }
        return PyLong_FromLong(rc);
    }
    static PyObject* call(PyObject*, PyObject* const* given, Py_ssize_t n) {
        if (n != (Py_ssize_t)sizeof...(A)) return PyErr_Format(PyExc_TypeError, "%s takes %zu arguments (%zd given)", name, sizeof...(A), n);
        return run(given, std::index_sequence_for<A...>{});
    }
};

#define SP_LAUNCHES(X)                                                                                                        \
    X(sp_gemm_abt) X(sp_gemm_abt_batched) X(sp_row_ops) X(sp_row_map_f32) X(sp_row_map_i32) X(sp_row_sample) X(sp_philox_uniforms) \
    X(sp_row_get_prob) X(sp_cem_resample) X(sp_cem_resample_philox) X(sp_row_reduce_f32) X(sp_cem_update_mask) X(sp_row_binarize)   \
    X(sp_map_f32) X(sp_reduce_sum) X(sp_reduce) X(sp_row_l1_normalize) X(sp_reduce_sum_static) X(sp_transpose_inner_b32)            \
    X(sp_mlp_forward) X(sp_mlp_pack_weights) X(sp_mlp_forward_packed) X(sp_mlp_forward_ensemble) X(sp_ensemble_binarize)            \
    X(sp_stack_forward_f32)

template <typename E>
bool bind_one(void* library, PyObject* functions, const char* name, PyMethodDef& def) {
    E::fn = (decltype(E::fn))dlsym(library, name);
    if (E::fn == nullptr) {
        PyErr_Format(PyExc_RuntimeError, "the library has no %s", name);
        return false;
    }
    E::name = name;
    if (E::self == nullptr) {
        def = PyMethodDef{name, (PyCFunction)(void (*)(void))&E::call, METH_FASTCALL, nullptr};
        E::self = PyCFunction_New(&def, nullptr);
        if (E::self == nullptr) return false;
    }
    return PyDict_SetItemString(functions, name, E::self) == 0;
}

// bind(path): a dict of the functions behind the library at `path`, which the process keeps (one library per process).
PyObject* bind(PyObject*, PyObject* path) {
    const char* p = PyUnicode_AsUTF8(path);
    if (p == nullptr) return nullptr;
    PyObject* ctypes = PyImport_ImportModule("ctypes");
    if (ctypes == nullptr) return nullptr;
    if (g_void_p == nullptr) g_void_p = PyObject_GetAttrString(ctypes, "c_void_p");
    if (g_void_p != nullptr && g_byref == nullptr) {
        PyObject* any = PyObject_CallMethod(ctypes, "c_int", nullptr);
        PyObject* ref = any != nullptr ? PyObject_CallMethod(ctypes, "byref", "O", any) : nullptr;
        if (ref != nullptr) {
            g_byref = (PyObject*)Py_TYPE(ref);
            Py_INCREF(g_byref);
            PyObject* const mro = Py_TYPE(any)->tp_mro;             // c_int, _SimpleCData, _CData, object
            g_cdata = PyTuple_GET_ITEM(mro, PyTuple_GET_SIZE(mro) - 2);
            Py_INCREF(g_cdata);
        }
        Py_XDECREF(ref);
        Py_XDECREF(any);
    }
    Py_DECREF(ctypes);
    if (g_void_p == nullptr || g_byref == nullptr) return nullptr;
    void* library = dlopen(p, RTLD_NOW | RTLD_LOCAL);
    if (library == nullptr) return PyErr_Format(PyExc_RuntimeError, "%s", dlerror());
    PyObject* functions = PyDict_New();
    if (functions == nullptr) return nullptr;
    bool ok = true;
    enum {
#define SP_ID(name) ID_##name,
        SP_LAUNCHES(SP_ID) COUNT
#undef SP_ID
    };
    static PyMethodDef defs[COUNT];
#define SP_BIND(name) ok = ok && bind_one<Entry<ID_##name, std::remove_pointer_t<decltype(&::name)>>>(library, functions, #name, defs[ID_##name]);
    SP_LAUNCHES(SP_BIND)
#undef SP_BIND
    if (!ok) {
        Py_DECREF(functions);
        return nullptr;
    }
    return functions;
}

// ptr(t, dtype=None, name="tensor"): the address of a contiguous ROCm tensor, None for None.
PyObject* ptr(PyObject*, PyObject* const* args, Py_ssize_t n, PyObject* keywords) {
    PyObject *t = n > 0 ? args[0] : nullptr, *dtype = n > 1 ? args[1] : Py_None, *name = n > 2 ? args[2] : nullptr;
    if (n > 3) return PyErr_Format(PyExc_TypeError, "ptr takes at most 3 arguments");
    for (Py_ssize_t i = 0; keywords != nullptr && i < PyTuple_GET_SIZE(keywords); ++i) {
        PyObject* key = PyTuple_GET_ITEM(keywords, i);
        if (PyUnicode_CompareWithASCIIString(key, "name") == 0) name = args[n + i];
        else if (PyUnicode_CompareWithASCIIString(key, "dtype") == 0) dtype = args[n + i];
        else if (PyUnicode_CompareWithASCIIString(key, "t") == 0) t = args[n + i];
        else return PyErr_Format(PyExc_TypeError, "ptr has no argument %U", key);
    }
    if (t == nullptr) return PyErr_Format(PyExc_TypeError, "ptr needs a tensor");
    if (t == Py_None) Py_RETURN_NONE;
    PyObject* const named = name;
    auto raise = [&](PyObject* type, const char* text) -> PyObject* {
        if (named != nullptr) return PyErr_Format(type, "%U %s", named, text);
        return PyErr_Format(type, "tensor %s", text);
    };
    try {
        if (!THPVariable_Check(t)) return raise(PyExc_TypeError, "must be a torch.Tensor");
        const at::Tensor& x = THPVariable_Unpack(t);
        if (!x.is_cuda()) return raise(PyExc_ValueError, ("must live on the GPU (got " + x.device().str() + ")").c_str());
        if (!x.is_contiguous()) return raise(PyExc_ValueError, "must be contiguous (row-major, innermost stride 1)");
        if (dtype != Py_None) {
            if (!THPDtype_Check(dtype)) return PyErr_Format(PyExc_TypeError, "dtype must be a torch.dtype");
            if (((THPDtype*)dtype)->scalar_type != x.scalar_type()) {
                PyObject* got = PyObject_GetAttrString(t, "dtype");
                if (got == nullptr) return nullptr;
                if (named != nullptr) PyErr_Format(PyExc_TypeError, "%U must have dtype %S, got %S", named, dtype, got);
                else PyErr_Format(PyExc_TypeError, "tensor must have dtype %S, got %S", dtype, got);
                Py_DECREF(got);
                return nullptr;
            }
        }
        void* const at = x.data_ptr();
        if (g_keep != nullptr && PyList_Append(g_keep, t) != 0) return nullptr;
        return PyLong_FromVoidPtr(at);
    } catch (const std::exception& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
        return nullptr;
    }
}

// tape(calls, keep): launches and tensors go into these lists from now on; tape(None, None): no longer.
PyObject* tape(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 2 || !((args[0] == Py_None && args[1] == Py_None) || (PyList_Check(args[0]) && PyList_Check(args[1]))))
        return PyErr_Format(PyExc_TypeError, "tape takes two lists, or None twice");
    PyObject *calls = args[0] == Py_None ? nullptr : args[0], *keep = args[1] == Py_None ? nullptr : args[1];
    Py_XINCREF(calls);
    Py_XINCREF(keep);
    std::swap(calls, g_calls);
    std::swap(keep, g_keep);
    Py_XDECREF(calls);
    Py_XDECREF(keep);
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {{"bind", bind, METH_O, nullptr},
                         {"ptr", (PyCFunction)(void (*)(void))ptr, METH_FASTCALL | METH_KEYWORDS, nullptr},
                         {"tape", (PyCFunction)(void (*)(void))tape, METH_FASTCALL, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "spiral_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_spiral_host() { return PyModule_Create(&module); }
