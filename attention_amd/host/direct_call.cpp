// Calls of the C ABI from Python without ctypes' per-argument objects: ctypes takes 3 to 4 us to pass the 20 arguments of a
// decode or forward call, as long as the whole launch of a short kernel; this takes a few hundred nanoseconds.
//
// bind(name, address, slow) gives a callable for one function of include/ahpc_hip.h.  It takes the ordinary cases itself - every argument an
// int, a float or None, in the number the function has - and hands everything else (ctypes objects, wrong types, numbers that do
// not fit, keyword arguments) to `slow`, the ctypes function of the same name, which then accepts or refuses it as ever.  As with
// ctypes.CDLL the interpreter lock is released during the call.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstddef>
#include <cstring>
#include <tuple>
#include <type_traits>
#include <utility>

#include "ahpc_hip.h"

namespace {

struct Callable {
    PyObject_HEAD
    vectorcallfunc vectorcall;
    void* address;
    PyObject* slow;
    // 1: called, result in *out; 0: not an ordinary call
    int (*invoke)(void* address, PyObject* const* args, Py_ssize_t n, PyObject** out);
};

// One argument.  False: leave the call to ctypes.
template <typename T> bool take(PyObject* o, T* out) {
    if constexpr (std::is_pointer_v<T>) {
        if (o == Py_None) {
            *out = nullptr;
            return true;
        }
        if (!PyLong_CheckExact(o)) return false;
        const unsigned long long v = PyLong_AsUnsignedLongLong(o);
        if (v == (unsigned long long)-1 && PyErr_Occurred()) {
            PyErr_Clear();
            return false;
        }
        *out = reinterpret_cast<T>(v);
        return true;
    } else if constexpr (std::is_floating_point_v<T>) {
        if (!PyFloat_Check(o)) return false;
        *out = (T)PyFloat_AS_DOUBLE(o);
        return true;
    } else {
        if (!PyLong_CheckExact(o)) return false;
        int overflow = 0;
        const long long v = PyLong_AsLongLongAndOverflow(o, &overflow);
        if (overflow || (std::is_unsigned_v<T> && v < 0) || (long long)(T)v != v) return false;
        *out = (T)v;
        return true;
    }
}

template <typename F> struct Signature;
template <typename R, typename... A> struct Signature<R(A...)> {
    template <size_t... I> static int call(void* address, PyObject* const* args, PyObject** out, std::index_sequence<I...>) {
        std::tuple<A...> a;
        if (!(take<A>(args[I], &std::get<I>(a)) && ...)) return 0;
        R r;
        Py_BEGIN_ALLOW_THREADS
        r = reinterpret_cast<R (*)(A...)>(address)(std::get<I>(a)...);
        Py_END_ALLOW_THREADS
        *out = std::is_unsigned_v<R> ? PyLong_FromUnsignedLongLong((unsigned long long)r) : PyLong_FromLongLong((long long)r);
        return 1;
    }
    static int invoke(void* address, PyObject* const* args, Py_ssize_t n, PyObject** out) {
        return n == (Py_ssize_t)sizeof...(A) ? call(address, args, out, std::index_sequence_for<A...>{}) : 0;
    }
};

struct Entry {
    const char* name;
    int (*invoke)(void*, PyObject* const*, Py_ssize_t, PyObject**);
};
#define ENTRY(f) {#f, &Signature<std::remove_pointer_t<decltype(&f)>>::invoke}
const Entry kEntries[] = {
    ENTRY(ahpc_hip_flash_fwd), ENTRY(ahpc_hip_flash_fwd_gqa), ENTRY(ahpc_hip_flash_fwd_masked), ENTRY(ahpc_hip_flash_fwd_varlen),
    ENTRY(ahpc_hip_flash_fwd_varlen_gqa), ENTRY(ahpc_hip_flash_bwd), ENTRY(ahpc_hip_flash_bwd_kept), ENTRY(ahpc_hip_flash_bwd_varlen),
    ENTRY(ahpc_hip_kv_scatter), ENTRY(ahpc_hip_kv_scatter_batch), ENTRY(ahpc_hip_kv_gather), ENTRY(ahpc_hip_paged_decode),
    ENTRY(ahpc_hip_paged_decode_gqa), ENTRY(ahpc_hip_paged_decode_noalloc),
};
#undef ENTRY

PyObject* callable_call(PyObject* self, PyObject* const* args, size_t nargsf, PyObject* names) {
    auto* c = reinterpret_cast<Callable*>(self);
    PyObject* out = nullptr;
    if (!names && c->invoke(c->address, args, PyVectorcall_NARGS(nargsf), &out)) return out;
    return PyObject_Vectorcall(c->slow, args, nargsf, names);
}
void callable_dealloc(PyObject* self) {
    Py_XDECREF(reinterpret_cast<Callable*>(self)->slow);
    Py_TYPE(self)->tp_free(self);
}
// argtypes, restype and the like are the ctypes function's
PyObject* callable_getattro(PyObject* self, PyObject* name) { return PyObject_GetAttr(reinterpret_cast<Callable*>(self)->slow, name); }

PyTypeObject CallableType = {PyVarObject_HEAD_INIT(nullptr, 0)};

PyObject* bind(PyObject*, PyObject* args) {
    const char* name;
    unsigned long long address;
    PyObject* slow;
    if (!PyArg_ParseTuple(args, "sKO", &name, &address, &slow)) return nullptr;
    for (const Entry& e : kEntries)
        if (!std::strcmp(e.name, name)) {
            Callable* c = PyObject_New(Callable, &CallableType);
            if (!c) return nullptr;
            c->vectorcall = callable_call;
            c->address = reinterpret_cast<void*>(address);
            Py_INCREF(slow);
            c->slow = slow;
            c->invoke = e.invoke;
            return reinterpret_cast<PyObject*>(c);
        }
    Py_INCREF(slow);  // functions that are not called often enough to matter
    return slow;
}

PyMethodDef kMethods[] = {{"bind", bind, METH_VARARGS, "bind(name, address, slow): a callable for one function of the C ABI"}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_direct_call", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__direct_call() {
    CallableType.tp_name = "attention_amd._direct_call.Callable";
    CallableType.tp_basicsize = sizeof(Callable);
    CallableType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL;
    CallableType.tp_vectorcall_offset = offsetof(Callable, vectorcall);
    CallableType.tp_call = PyVectorcall_Call;
    CallableType.tp_dealloc = callable_dealloc;
    CallableType.tp_getattro = callable_getattro;
    if (PyType_Ready(&CallableType) < 0) return nullptr;
    return PyModule_Create(&kModule);
}
