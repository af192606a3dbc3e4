// Calls into libfastdl_gemm.so for fast_dl_amd.capi without ctypes' per-argument
// conversion objects.  A GEMM's 22 arguments cost ctypes 2.4 us per call and
// its Python wrapper 1.0 us more, as long as a small kernel runs; here they
// cost 0.4 us (measured on no-op calls, one core).
//
// The entry points' addresses come from capi.load_library(), so importing this
// module loads nothing.  Anything out of the ordinary -- the library not yet
// loaded, an argument that is not a plain int, float or None, or does not fit
// its C type -- goes to the ctypes binding, which treats it as it always did.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <fastdl_data.h>
#include <fastdl_gemm.h>

#include <cstdint>
#include <cstring>
#include <limits>
#include <tuple>
#include <type_traits>
#include <utility>

namespace {

// One C argument from a Python one; false: leave the call to ctypes.
template <class T>
bool convert(PyObject* o, T& out) {
    if constexpr (std::is_pointer_v<T>) {
        if (o == Py_None) {
            out = nullptr;
            return true;
        }
        if (!PyLong_CheckExact(o)) return false;
        const unsigned long long v = PyLong_AsUnsignedLongLong(o);
        if (v == ~0ull && PyErr_Occurred()) {
            PyErr_Clear();
            return false;
        }
        out = reinterpret_cast<T>(static_cast<uintptr_t>(v));
        return true;
    } else if constexpr (std::is_floating_point_v<T>) {
        if (!PyFloat_CheckExact(o)) return false;
        out = static_cast<T>(PyFloat_AS_DOUBLE(o));
        return true;
    } else if constexpr (std::is_signed_v<T>) {
        if (!PyLong_CheckExact(o)) return false;
        int overflow = 0;
        const long long v = PyLong_AsLongLongAndOverflow(o, &overflow);
        if (overflow || v < (long long)std::numeric_limits<T>::min() ||
            v > (long long)std::numeric_limits<T>::max()) {
            return false;
        }
        out = static_cast<T>(v);
        return true;
    } else {
        if (!PyLong_CheckExact(o)) return false;
        const unsigned long long v = PyLong_AsUnsignedLongLong(o);
        if (v == ~0ull && PyErr_Occurred()) {
            PyErr_Clear();
            return false;
        }
        out = static_cast<T>(v);
        return true;
    }
}

// An entry point: its address once the library is loaded, the ctypes call and
// the function that raises for a non-zero status.
struct Entry {
    void* address = nullptr;
    PyObject* slow = nullptr;
    PyObject* fail = nullptr;
};

template <class F, int Id>
struct Call;

template <class... A, int Id>
struct Call<int (*)(A...), Id> {
    static inline Entry entry;
    static inline const char* name = "";

    template <size_t... I>
    static PyObject* run(PyObject* const* args, Py_ssize_t n, std::index_sequence<I...>) {
        std::tuple<A...> v;
        if (!entry.address || n != (Py_ssize_t)sizeof...(A) ||
            !(convert(args[I], std::get<I>(v)) && ...)) {
            return PyObject_Vectorcall(entry.slow, args, (size_t)n, nullptr);
        }
        int status;
        Py_BEGIN_ALLOW_THREADS
        status = reinterpret_cast<int (*)(A...)>(entry.address)(std::get<I>(v)...);
        Py_END_ALLOW_THREADS
        if (status != 0) return PyObject_CallFunction(entry.fail, "si", name, status);
        return PyLong_FromLong(0);
    }

    static PyObject* fast(PyObject*, PyObject* const* args, Py_ssize_t n) {
        return run(args, n, std::index_sequence_for<A...>{});
    }
};

struct Bound {
    const char* name;
    Entry* entry;
    PyMethodDef def;
};

template <class C>
Bound bound(const char* name) {
    C::name = name;
    return {name, &C::entry,
            {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(&C::fast)),
             METH_FASTCALL, nullptr}};
}

#define FDL_BOUND(FN) bound<Call<decltype(&FN), __LINE__>>(#FN)
Bound g_bound[] = {
    FDL_BOUND(fdl_sgemm_ex),
    FDL_BOUND(fdl_sgemm_ex_select),
    FDL_BOUND(fdl_sgemm_ex_ws),
    FDL_BOUND(fdl_sgemm_ex_noalloc),
    FDL_BOUND(fdl_gemm),
    FDL_BOUND(fdl_add_row_bias),
    FDL_BOUND(fdl_relu),
    FDL_BOUND(fdl_relu_backward),
    FDL_BOUND(fdl_colsum),
    FDL_BOUND(fdl_softmax),
    FDL_BOUND(fdl_softmax_xent),
    FDL_BOUND(fdl_sgd_update),
    FDL_BOUND(fdl_mlp2_train_step),
    FDL_BOUND(fdl_idx_gather),
};

Bound* find(const char* name) {
    for (Bound& b : g_bound) {
        if (strcmp(b.name, name) == 0) return &b;
    }
    return nullptr;
}

// bind(name, slow, fail) -> the callable for an entry point, or None if this
// module has none.
PyObject* py_bind(PyObject*, PyObject* args) {
    const char* name;
    PyObject *slow, *fail;
    if (!PyArg_ParseTuple(args, "sOO", &name, &slow, &fail)) return nullptr;
    Bound* b = find(name);
    if (!b) Py_RETURN_NONE;
    Py_INCREF(slow);
    Py_INCREF(fail);
    Py_XSETREF(b->entry->slow, slow);
    Py_XSETREF(b->entry->fail, fail);
    return PyCFunction_New(&b->def, nullptr);
}

// set_address(name, address): the entry point in the loaded library.
PyObject* py_set_address(PyObject*, PyObject* args) {
    const char* name;
    unsigned long long address;
    if (!PyArg_ParseTuple(args, "sK", &name, &address)) return nullptr;
    if (Bound* b = find(name)) b->entry->address = reinterpret_cast<void*>((uintptr_t)address);
    Py_RETURN_NONE;
}

PyMethodDef g_methods[] = {{"bind", py_bind, METH_VARARGS, nullptr},
                           {"set_address", py_set_address, METH_VARARGS, nullptr},
                           {nullptr, nullptr, 0, nullptr}};

PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_fastcall", nullptr, -1, g_methods,
                        nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fastcall() { return PyModule_Create(&g_module); }
