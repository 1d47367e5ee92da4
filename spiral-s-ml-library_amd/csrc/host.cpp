// The host path of a call: device pointers of tensors and launches of the C-ABI library without ctypes.
//
// A small kernel takes 2 to 4 us, and with ctypes a call took 6.5 to 10 us of host: about 0.7 us for the checks and the address of each
// tensor in Python, and 2 us to convert the arguments.  Both are done here; bind() makes a function of every entry point that launches
// work, from its own declaration in spiral_mi355.h, and an argument has to be of the declared type.  (us a call with the queue kept full, ctypes
// / here: a four-layer stack on packed weights 7.2 / 5.6, one on row-major weights 11.4 / 7.1, the CEM update 76 / 63, a GEMM of 16 x 16 x 296
// 7.6 / 5.4, a sampled softmax of 32 rows with its outputs allocated 11.7 / 8.7.)  What is left is the runtime's launch, about 4 us.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include <dlfcn.h>
#include <string.h>

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
PyObject* g_void_p = nullptr;     // of ctypes: c_void_p, c_int32, Array, _Pointer, cast, the type of byref(...)
PyObject* g_int32 = nullptr;
PyObject* g_array = nullptr;
PyObject* g_pointer = nullptr;
PyObject* g_cast = nullptr;
PyObject* g_byref = nullptr;

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
        p = (void*)PyLong_AsUnsignedLongLongMask(o);      // as ctypes: the low bits
        return true;
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

// The buffer behind an object of ctypes.
struct Buffer {
    Py_buffer view{};
    Buffer() = default;
    Buffer(const Buffer&) = delete;
    ~Buffer() {
        if (view.obj != nullptr) PyBuffer_Release(&view);
    }
    bool take(PyObject* o) { return PyObject_GetBuffer(o, &view, PyBUF_SIMPLE) == 0; }
};

bool refuse(PyObject* o, const char* what) {
    PyErr_Format(PyExc_TypeError, "%s, not %s", what, Py_TYPE(o)->tp_name);
    return false;
}

// Whether `o` is a ctypes array of `element`, or a ctypes pointer to it (`base`: ctypes.Array, ctypes._Pointer); -1 with an exception.
int is_of(PyObject* o, PyObject* base, PyObject* element) {
    const int is_base = PyObject_IsInstance(o, base);
    if (is_base <= 0) return is_base;
    PyObject* type = PyObject_GetAttrString((PyObject*)Py_TYPE(o), "_type_");
    if (type == nullptr) return -1;
    Py_DECREF(type);
    return type == element;
}

// The address that a ctypes pointer object holds.
bool pointed_to(PyObject* o, void*& p) {
    Buffer own;
    if (!own.take(o)) return false;
    p = *(void**)own.view.buf;
    return true;
}

// byref(x): x, if it is an instance of `type` and the reference is to its start; nullptr with an exception if not.
PyObject* referred(PyObject* o, PyObject* type, const char* what) {
    PyObject* target = PyObject_GetAttrString(o, "_obj");
    if (target == nullptr) return nullptr;
    Buffer own;
    PyObject* at = nullptr;
    const bool fits = PyObject_TypeCheck(target, (PyTypeObject*)type) != 0;
    if (fits && own.take(target)) {
        PyObject* address = PyObject_CallFunctionObjArgs(g_cast, o, g_void_p, nullptr);
        at = address != nullptr ? PyObject_GetAttrString(address, "value") : nullptr;
        Py_XDECREF(address);
    }
    const bool start = at != nullptr && at != Py_None && PyLong_AsVoidPtr(at) == own.view.buf;
    Py_XDECREF(at);
    if (!start) {
        if (!PyErr_Occurred()) {
            if (fits) PyErr_Format(PyExc_TypeError, "%s, not a reference with an offset", what);
            else PyErr_Format(PyExc_TypeError, "%s, not a reference to %s", what, Py_TYPE(target)->tp_name);
        }
        Py_DECREF(target);
        return nullptr;
    }
    return target;
}

// Scalars may come as objects of ctypes, of the parameter's own type.
PyObject* g_scalars[5] = {};      // c_int32, c_int64, c_uint32, c_uint64, c_float
const char* const SCALARS[5] = {"c_int32", "c_int64", "c_uint32", "c_uint64", "c_float"};
template <typename T>
PyObject* scalar_type() {
    return g_scalars[std::is_floating_point_v<T> ? 4 : 2 * std::is_unsigned_v<T> + (sizeof(T) == 8)];
}
template <typename Take>
bool unwrapped(PyObject* o, PyObject* type, const Take& take) {
    if (!PyObject_TypeCheck(o, (PyTypeObject*)type)) return take(o);
    PyObject* v = PyObject_GetAttrString(o, "value");
    if (v == nullptr) return false;
    const bool ok = take(v);
    Py_DECREF(v);
    return ok;
}

// What a function is bound to, in a capsule that the function object holds.
struct Bound {
    void* fn;
    PyObject* stream;             // the ctypes structure that stands for sp_philox_t
    const char* name;
    PyObject* function = nullptr; // the function object itself: what the tape records
    Bound(void* fn, PyObject* stream, const char* name) : fn(fn), stream(Py_NewRef(stream)), name(name) {}
    Bound(const Bound&) = delete;
    ~Bound() { Py_DECREF(stream); }
};

// HOST_INTS: of an entry point whose const int32_t* are host arrays.  Those that take arrays of addresses take the widths of a stack
// beside them; everywhere else a const int32_t* is device memory.
template <typename T, bool HOST_INTS, typename = void>
struct Arg;

template <typename T, bool HOST_INTS>
struct Arg<T, HOST_INTS, std::enable_if_t<std::is_integral_v<T>>> {
    T value = 0;
    bool load(PyObject* o, const Bound&) {
        unsigned long long v = 0;
        if (PyLong_Check(o) ? !as_integer(o, v) : !unwrapped(o, scalar_type<T>(), [&](PyObject* x) { return as_integer(x, v); })) return false;
        value = (T)v;
        return true;
    }
};

template <typename T, bool HOST_INTS>
struct Arg<T, HOST_INTS, std::enable_if_t<std::is_floating_point_v<T>>> {
    T value = 0;
    bool load(PyObject* o, const Bound&) {
        double v = 0;
        auto number = [&](PyObject* x) {
            v = PyFloat_AsDouble(x);
            return !(v == -1.0 && PyErr_Occurred());
        };
        if (PyFloat_Check(o) ? !number(o) : !unwrapped(o, scalar_type<T>(), number)) return false;
        value = (T)v;
        return true;
    }
};

// Device memory: an address, or a ctypes pointer that holds one.
template <typename T, bool HOST_INTS>
struct Arg<T*, HOST_INTS, std::enable_if_t<!std::is_pointer_v<std::remove_const_t<T>> && !std::is_same_v<T, const sp_philox_t> &&
                                           !(HOST_INTS && std::is_same_v<T, const int32_t>)>> {
    T* value = nullptr;
    bool load(PyObject* o, const Bound&) {
        void* p = nullptr;
        if (o != Py_None && !PyLong_Check(o)) {
            const int is_pointer = PyObject_IsInstance(o, g_pointer);
            if (is_pointer < 0 || (is_pointer > 0 ? !pointed_to(o, p) : !as_address(o, p))) return false;
        } else if (!as_address(o, p)) {
            return false;
        }
        value = (T*)p;
        return true;
    }
};

// A host array of addresses or of 32-bit integers: a list, a tuple, or of ctypes an array of such elements, one of them by reference or a
// pointer to them.  Elements are copied, zeros behind them, so that what reads further than was given -- a stack has eight layers at
// most -- finds zeros; only longer arrays, and what a pointer points to, are read in place.
template <typename T, bool HOST_INTS>
struct Arg<T*, HOST_INTS, std::enable_if_t<std::is_pointer_v<std::remove_const_t<T>> || (HOST_INTS && std::is_same_v<T, const int32_t>)>> {
    typedef std::remove_const_t<T> Element;
    static constexpr bool ADDRESSES = std::is_pointer_v<Element>;
    T* value = nullptr;
    Element few[MOST] = {};
    std::unique_ptr<Element[]> many;
    Buffer buffer;

    bool list(PyObject* o) {
        const Py_ssize_t n = PySequence_Fast_GET_SIZE(o);
        Element* elements = few;
        if (n > MOST) {
            many.reset(new (std::nothrow) Element[n]);
            elements = many.get();
            if (elements == nullptr) {
                PyErr_NoMemory();
                return false;
            }
        }
        for (Py_ssize_t i = 0; i < n; ++i) {
            if (i >= PySequence_Fast_GET_SIZE(o)) {        // (an element's __index__ may shorten the list)
                PyErr_SetString(PyExc_RuntimeError, "a list of arguments changed its size");
                return false;
            }
            PyObject* e = Py_NewRef(PySequence_Fast_GET_ITEM(o, i));
            bool ok;
            if constexpr (ADDRESSES) {
                void* p = nullptr;
                ok = as_address(e, p);
                elements[i] = (Element)p;
            } else {
                unsigned long long v = 0;
                ok = as_integer(e, v);
                elements[i] = (Element)v;
            }
            Py_DECREF(e);
            if (!ok) return false;
        }
        value = elements;
        return true;
    }
    bool memory(PyObject* o) {                             // of an array, or of one element
        if (!buffer.take(o)) return false;
        const size_t n = (size_t)buffer.view.len / sizeof(Element);
        if (n <= (size_t)MOST) memcpy(few, buffer.view.buf, n * sizeof(Element));
        value = n <= (size_t)MOST ? few : (T*)buffer.view.buf;
        return true;
    }
    bool load(PyObject* o, const Bound&) {
        if (PyTuple_Check(o) || PyList_Check(o)) return list(o);
        if (o == Py_None) return true;
        PyObject* const type = ADDRESSES ? g_void_p : g_int32;
        const char* const what = ADDRESSES ? "an array of addresses is None, a list, a tuple or of c_void_p" : "an array of integers is None, a list, a tuple or of c_int32";
        const int is_array = is_of(o, g_array, type);
        if (is_array != 0) return is_array > 0 && memory(o);
        const int is_pointer = is_of(o, g_pointer, type);
        if (is_pointer != 0) {
            void* p = nullptr;
            if (is_pointer < 0 || !pointed_to(o, p)) return false;
            value = (T*)p;
            return true;
        }
        if ((PyObject*)Py_TYPE(o) == g_byref) {
            PyObject* target = referred(o, type, what);
            if (target == nullptr) return false;
            const bool ok = memory(target);
            Py_DECREF(target);
            return ok;
        }
        return refuse(o, what);
    }
};

// The state of a random stream, a host structure: the structure, a reference or a ctypes pointer to it, or an array of them.
template <bool HOST_INTS>
struct Arg<const sp_philox_t*, HOST_INTS> {
    const sp_philox_t* value = nullptr;
    Buffer buffer;
    bool memory(PyObject* o) {
        if (!buffer.take(o)) return false;
        if ((size_t)buffer.view.len < sizeof(sp_philox_t)) return refuse(o, "a random stream needs a whole PhiloxConfig");
        value = (const sp_philox_t*)buffer.view.buf;
        return true;
    }
    bool load(PyObject* o, const Bound& bound) {
        if (o == Py_None) return true;
        if (PyObject_TypeCheck(o, (PyTypeObject*)bound.stream)) return memory(o);
        const char* const what = "a random stream is None or a PhiloxConfig";
        if ((PyObject*)Py_TYPE(o) == g_byref) {
            PyObject* target = referred(o, bound.stream, what);
            if (target == nullptr) return false;
            const bool ok = memory(target);
            Py_DECREF(target);
            return ok;
        }
        const int is_array = is_of(o, g_array, bound.stream);
        if (is_array != 0) return is_array > 0 && memory(o);
        const int is_pointer = is_of(o, g_pointer, bound.stream);
        if (is_pointer == 0) return refuse(o, what);
        void* p = nullptr;
        if (is_pointer < 0 || !pointed_to(o, p)) return false;
        value = (const sp_philox_t*)p;
        return true;
    }
};

// What does not fit is reported as ctypes reports it; as a TypeError, too.
PyObject* g_argument_error = nullptr;
void refuse_argument(int number) {
    if (!PyErr_ExceptionMatches(PyExc_TypeError)) return;
    PyObject *type, *text, *trace;
    PyErr_Fetch(&type, &text, &trace);
    PyErr_Format(g_argument_error, "argument %d: %S", number, text != nullptr ? text : Py_None);
    Py_XDECREF(type);
    Py_XDECREF(text);
    Py_XDECREF(trace);
}

// ---- one function per entry point ----
template <typename F>
struct Entry;
template <typename... A>
struct Entry<int(A...)> {
    static constexpr bool HOST_INTS = ((std::is_pointer_v<A> && std::is_pointer_v<std::remove_const_t<std::remove_pointer_t<A>>>) || ...);

    template <size_t... I>
    static PyObject* run(const Bound& bound, PyObject* const* given, std::index_sequence<I...>) {
        std::tuple<Arg<A, HOST_INTS>...> args;
        if (int at = 0; !((++at, std::get<I>(args).load(given[I], bound)) && ...)) {
            refuse_argument(at);
            return nullptr;
        }
        int (*const fn)(A...) = (int (*)(A...))bound.fn;
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
            PyObject* call = PyTuple_Pack(2, bound.function, kept);
            Py_DECREF(kept);
            if (call == nullptr) return nullptr;
            const int failed = PyList_Append(g_calls, call);
            Py_DECREF(call);
            if (failed != 0) return nullptr;
        }
        return PyLong_FromLong(rc);
    }
    static PyObject* call(PyObject* capsule, PyObject* const* given, Py_ssize_t n) {
        const Bound* const bound = (const Bound*)PyCapsule_GetPointer(capsule, nullptr);
        if (bound == nullptr) return nullptr;
        if (n != (Py_ssize_t)sizeof...(A)) return PyErr_Format(PyExc_TypeError, "%s takes %zu arguments (%zd given)", bound->name, sizeof...(A), n);
        return run(*bound, given, std::index_sequence_for<A...>{});
    }
};

#define SP_LAUNCHES(X)                                                                                                        \
    X(sp_gemm_abt) X(sp_gemm_abt_batched) X(sp_row_ops) X(sp_row_map_f32) X(sp_row_map_i32) X(sp_row_sample) X(sp_philox_uniforms) \
    X(sp_row_get_prob) X(sp_cem_resample) X(sp_cem_resample_philox) X(sp_row_reduce_f32) X(sp_cem_update_mask) X(sp_row_binarize)   \
    X(sp_map_f32) X(sp_reduce_sum) X(sp_reduce) X(sp_row_l1_normalize) X(sp_reduce_sum_static) X(sp_transpose_inner_b32)            \
    X(sp_mlp_forward) X(sp_mlp_pack_weights) X(sp_mlp_forward_packed) X(sp_mlp_forward_ensemble) X(sp_ensemble_binarize)            \
    X(sp_stack_forward_f32)

bool bind_one(void* library, PyObject* stream, PyObject* functions, const char* name, PyCFunction call, PyMethodDef& def) {
    void* const fn = dlsym(library, name);
    if (fn == nullptr) {
        PyErr_Format(PyExc_RuntimeError, "the library has no %s", name);
        return false;
    }
    def = PyMethodDef{name, call, METH_FASTCALL, nullptr};
    Bound* const bound = new (std::nothrow) Bound(fn, stream, name);
    if (bound == nullptr) {
        PyErr_NoMemory();
        return false;
    }
    PyObject* capsule = PyCapsule_New(bound, nullptr, [](PyObject* c) { delete (Bound*)PyCapsule_GetPointer(c, nullptr); });
    if (capsule == nullptr) {
        delete bound;
        return false;
    }
    PyObject* function = PyCFunction_New(&def, capsule);
    Py_DECREF(capsule);
    if (function == nullptr) return false;
    bound->function = function;                            // (borrowed: the function holds the capsule)
    const int failed = PyDict_SetItemString(functions, name, function);
    Py_DECREF(function);
    return failed == 0;
}

// bind(path, stream): a dict of the functions behind the library at `path`, which the process keeps; `stream`: the ctypes structure
// that stands for sp_philox_t in their calls.
PyObject* bind(PyObject*, PyObject* const* given, Py_ssize_t n) {
    if (n != 2 || !PyType_Check(given[1])) return PyErr_Format(PyExc_TypeError, "bind takes a path and a structure type");
    const char* p = PyUnicode_AsUTF8(given[0]);
    if (p == nullptr) return nullptr;
    PyObject* ctypes = PyImport_ImportModule("ctypes");
    if (ctypes == nullptr) return nullptr;
    auto get = [&](PyObject*& to, const char* name) { return to != nullptr || (to = PyObject_GetAttrString(ctypes, name)) != nullptr; };
    bool found = get(g_void_p, "c_void_p") && get(g_int32, "c_int32") && get(g_array, "Array") && get(g_pointer, "_Pointer") && get(g_cast, "cast");
    for (int i = 0; i < 5; ++i) found = found && get(g_scalars[i], SCALARS[i]);
    if (found && g_byref == nullptr) {
        PyObject* any = PyObject_CallMethod(ctypes, "c_int", nullptr);
        PyObject* ref = any != nullptr ? PyObject_CallMethod(ctypes, "byref", "O", any) : nullptr;
        if (ref != nullptr) g_byref = Py_NewRef((PyObject*)Py_TYPE(ref));
        Py_XDECREF(ref);
        Py_XDECREF(any);
        found = g_byref != nullptr;
    }
    if (found && g_argument_error == nullptr) {
        PyObject* of_ctypes = PyObject_GetAttrString(ctypes, "ArgumentError");
        PyObject* bases = of_ctypes != nullptr ? PyTuple_Pack(2, of_ctypes, PyExc_TypeError) : nullptr;
        g_argument_error = bases != nullptr ? PyErr_NewException("spiral_host.ArgumentError", bases, nullptr) : nullptr;
        Py_XDECREF(bases);
        Py_XDECREF(of_ctypes);
        found = g_argument_error != nullptr;
    }
    Py_DECREF(ctypes);
    if (!found) return nullptr;
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
#define SP_BIND(name) ok = ok && bind_one(library, given[1], functions, #name, (PyCFunction)(void (*)(void))&Entry<std::remove_pointer_t<decltype(&::name)>>::call, defs[ID_##name]);
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
        else return PyErr_Format(PyExc_TypeError, "ptr has no argument %S", key);
    }
    if (t == nullptr) return PyErr_Format(PyExc_TypeError, "ptr needs a tensor");
    if (t == Py_None) Py_RETURN_NONE;
    PyObject* const named = name;
    auto raise = [&](PyObject* type, const char* text) -> PyObject* {
        if (named != nullptr) return PyErr_Format(type, "%S %s", named, text);
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
                if (named != nullptr) PyErr_Format(PyExc_TypeError, "%S must have dtype %S, got %S", named, dtype, got);
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

PyMethodDef methods[] = {{"bind", (PyCFunction)(void (*)(void))bind, METH_FASTCALL, nullptr},
                         {"ptr", (PyCFunction)(void (*)(void))ptr, METH_FASTCALL | METH_KEYWORDS, nullptr},
                         {"tape", (PyCFunction)(void (*)(void))tape, METH_FASTCALL, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "spiral_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_spiral_host() { return PyModule_Create(&module); }
