// CPython entry into the C ABI: `call(name, *args)` for the entry points whose arguments are numbers and
// pointers, and the operator table's lookup, without the per-argument objects of ctypes.
//
// What it saves: a product call has fifteen arguments, which ctypes converts one by one through Python-level
// descriptors before the launch; an operator of the Python surface is such a call, a lookup and an allocation.
// Calls take exactly int, float or None per argument; anything else (byref, arrays, numpy numbers, structures, another
// count of arguments) goes to the general ctypes path of lib.py, which also loads the library at the first call
// and raises for a failed status.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <stddef.h>
#include <string.h>

#include <tuple>
#include <type_traits>
#include <utility>

#include "../../include/minit_hip.h"

namespace {

// One argument; false where it is not the plain object the parameter's type takes.  Integers are reduced to the
// parameter's width as ctypes does.
template <class T>
bool convert(PyObject* o, T& v) {
    if constexpr (std::is_pointer_v<T>) {
        if (o == Py_None) {
            v = nullptr;
            return true;
        }
        if (!PyLong_CheckExact(o)) return false;
        v = reinterpret_cast<T>(PyLong_AsUnsignedLongMask(o));
    } else if constexpr (std::is_floating_point_v<T>) {
        if (!PyFloat_CheckExact(o)) return false;
        v = (T)PyFloat_AS_DOUBLE(o);
    } else {
        if (!PyLong_CheckExact(o)) return false;
        v = (T)PyLong_AsUnsignedLongMask(o);
    }
    return true;
}

// ctypes' code of a type (c_int._type_ and so on).
template <class T>
constexpr char code() {
    if constexpr (std::is_pointer_v<T>) return 'P';
    else if constexpr (std::is_same_v<T, double>) return 'd';
    else if constexpr (std::is_same_v<T, float>) return 'f';
    else if constexpr (std::is_same_v<T, int>) return 'i';
    else {
        static_assert(std::is_same_v<T, unsigned long>, "a type without a code");
        return 'L';
    }
}

// Thunk<decltype(f)>::run: converts, calls f with the interpreter lock released, leaves the result; false, and no
// call, where an argument is not plain.
template <class F>
struct Thunk;
template <class R, class... A>
struct Thunk<R(A...)> {
    static constexpr int kCount = sizeof...(A);
    static constexpr char kSignature[] = {code<R>(), code<A>()..., 0};
    template <size_t... I>
    static bool invoke(void* fn, PyObject* const* args, unsigned long* result, std::index_sequence<I...>) {
        [[maybe_unused]] std::tuple<A...> held;
        if (!(convert(args[I], std::get<I>(held)) && ...)) return false;
        R r;
        Py_BEGIN_ALLOW_THREADS
        r = reinterpret_cast<R (*)(A...)>(fn)(std::get<I>(held)...);
        Py_END_ALLOW_THREADS
        *result = (unsigned long)r;
        return true;
    }
    static bool run(void* fn, PyObject* const* args, unsigned long* result) {
        return invoke(fn, args, result, std::make_index_sequence<sizeof...(A)>());
    }
};

struct Entry {
    const char* name;
    bool (*run)(void*, PyObject* const*, unsigned long*);
    int count;
    const char* signature;   // codes of the result and the arguments
    bool status;   // the result is a status code: non-zero raises
    void* fn;      // set once the library is loaded
};

#define STATUS(f) {#f, Thunk<decltype(f)>::run, Thunk<decltype(f)>::kCount, Thunk<decltype(f)>::kSignature, true, nullptr}
#define SIZE(f) {#f, Thunk<decltype(f)>::run, Thunk<decltype(f)>::kCount, Thunk<decltype(f)>::kSignature, false, nullptr}
Entry g_entries[] = {
    STATUS(mh_free), STATUS(mh_memcpy), STATUS(mh_memset), STATUS(mh_stream_synchronize), STATUS(mh_device_synchronize),
    STATUS(mh_event_record), STATUS(mh_event_synchronize), STATUS(mh_copy_kernel), STATUS(mh_gptq_unpack),
    STATUS(mh_gptq_dequant), SIZE(mh_gptq_workspace_bytes), STATUS(mh_gptq_gemv), STATUS(mh_gptq_gemm),
    STATUS(mh_gptq_matmul), STATUS(mh_gptq_linear), STATUS(mh_gptq_matmul_static),
    SIZE(mh_gptq_silu_pairs_workspace_bytes), STATUS(mh_gptq_matmul_silu_pairs), STATUS(mh_f16_matmul_nk),
    STATUS(mh_f16_matmul_nk_batched), STATUS(mh_i8_gemm), STATUS(mh_i8_transpose), STATUS(mh_gptq_permute_rows),
    STATUS(mh_rms_norm), STATUS(mh_rope), STATUS(mh_softmax), STATUS(mh_softmax_causal), STATUS(mh_sum), STATUS(mh_max),
    STATUS(mh_mean), STATUS(mh_sigmoid), STATUS(mh_gather_columns), STATUS(mh_multiply), STATUS(mh_add),
    STATUS(mh_silu_mul), STATUS(mh_add_bias), STATUS(mh_add_rms_norm), STATUS(mh_argmax),
    SIZE(mh_attn_decode_workspace_bytes), STATUS(mh_attn_decode), STATUS(mh_rope_kv_append),
};
#undef STATUS
#undef SIZE

PyObject* g_table = nullptr;     // name -> capsule of its entry, filled by bind()
PyObject* g_general = nullptr;   // lib.py: the ctypes path
PyObject* g_failed = nullptr;    // lib.py: raises for (name, status)

PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t n) {
    PyObject* found = n > 0 && g_table != nullptr ? PyDict_GetItemWithError(g_table, args[0]) : nullptr;
    if (found != nullptr) {
        const Entry* e = static_cast<Entry*>(PyLong_AsVoidPtr(found));
        unsigned long r = 0;
        if (n - 1 == e->count && e->run(e->fn, args + 1, &r)) {
            if (!e->status) return PyLong_FromUnsignedLong(r);
            if ((int)r == 0) return PyLong_FromLong(0);
            return PyObject_CallFunction(g_failed, "Oi", args[0], (int)r);
        }
    } else if (PyErr_Occurred()) {
        return nullptr;
    }
    if (g_general == nullptr) {
        PyErr_SetString(PyExc_RuntimeError, "binding: set_hooks() has not been called");
        return nullptr;
    }
    return PyObject_Vectorcall(g_general, args, (size_t)n, nullptr);
}

PyObject* set_hooks(PyObject*, PyObject* args) {
    PyObject *general, *failed;
    if (!PyArg_ParseTuple(args, "OO", &general, &failed)) return nullptr;
    Py_INCREF(general);
    Py_INCREF(failed);
    Py_XSETREF(g_general, general);
    Py_XSETREF(g_failed, failed);
    Py_RETURN_NONE;
}

// bind({name: (address, signature)}): the entry points of a loaded library.  One whose signature is another than the header
// had when this module was compiled is left to the ctypes path: the two may come from different builds.  Returns how many.
PyObject* bind(PyObject*, PyObject* entries) {
    if (!PyDict_Check(entries)) {
        PyErr_SetString(PyExc_TypeError, "bind: a dict of addresses and signatures is expected");
        return nullptr;
    }
    PyObject* table = PyDict_New();
    if (table == nullptr) return nullptr;
    long left = 0;
    for (Entry& e : g_entries) {
        PyObject *given = PyDict_GetItemString(entries, e.name), *address;
        if (given == nullptr) continue;
        const char* signature;
        void* fn = nullptr;
        PyObject* entry = nullptr;
        if (PyArg_ParseTuple(given, "Os", &address, &signature)) {
            if (strcmp(signature, e.signature) != 0) {
                ++left;
                continue;
            }
            fn = PyLong_AsVoidPtr(address);
            entry = PyErr_Occurred() ? nullptr : PyLong_FromVoidPtr(&e);
        }
        PyObject* name = entry != nullptr ? PyUnicode_InternFromString(e.name) : nullptr;
        const bool stored = name != nullptr && PyDict_SetItem(table, name, entry) == 0;
        Py_XDECREF(entry);
        Py_XDECREF(name);
        if (!stored) {
            Py_DECREF(table);
            return nullptr;
        }
        e.fn = fn;
    }
    Py_XSETREF(g_table, table);
    return PyLong_FromLong(left);
}

// dispatcher(cache, lookup) -> dispatch(*args): cache[tuple(arg.type() for arg in args)](*args), the
// implementation looked up (and cached) by lookup(types) where it is missing.
struct Dispatcher {
    PyObject_HEAD
    PyObject* cache;
    PyObject* lookup;
    vectorcallfunc vectorcall;
};
PyObject* g_type_name = nullptr;   // "type"

PyObject* dispatch_call(PyObject* self, PyObject* const* args, size_t nargsf, PyObject* kwnames) {
    Dispatcher* d = reinterpret_cast<Dispatcher*>(self);
    const Py_ssize_t n = PyVectorcall_NARGS(nargsf);
    if (kwnames != nullptr && PyTuple_GET_SIZE(kwnames) > 0) {
        PyErr_SetString(PyExc_TypeError, "dispatch takes no keyword arguments");
        return nullptr;
    }
    PyObject* types = PyTuple_New(n);
    if (types == nullptr) return nullptr;
    for (Py_ssize_t i = 0; i < n; ++i) {
        PyObject* t = PyObject_CallMethodNoArgs(args[i], g_type_name);
        if (t == nullptr) {
            Py_DECREF(types);
            return nullptr;
        }
        PyTuple_SET_ITEM(types, i, t);
    }
    PyObject* func = PyDict_GetItemWithError(d->cache, types);
    if (func != nullptr) {
        Py_INCREF(func);
    } else if (!PyErr_Occurred()) {
        func = PyObject_CallOneArg(d->lookup, types);
        if (func != nullptr && PyDict_SetItem(d->cache, types, func) < 0) Py_CLEAR(func);
    }
    Py_DECREF(types);
    if (func == nullptr) return nullptr;
    PyObject* result = PyObject_Vectorcall(func, args, (size_t)n, nullptr);
    Py_DECREF(func);
    return result;
}

void dispatcher_dealloc(PyObject* self) {
    Dispatcher* d = reinterpret_cast<Dispatcher*>(self);
    Py_XDECREF(d->cache);
    Py_XDECREF(d->lookup);
    Py_TYPE(self)->tp_free(self);
}

PyTypeObject g_dispatcher_type = {PyVarObject_HEAD_INIT(nullptr, 0)};

PyObject* dispatcher(PyObject*, PyObject* args) {
    PyObject *cache, *lookup;
    if (!PyArg_ParseTuple(args, "O!O", &PyDict_Type, &cache, &lookup)) return nullptr;
    Dispatcher* d = PyObject_New(Dispatcher, &g_dispatcher_type);
    if (d == nullptr) return nullptr;
    Py_INCREF(cache);
    Py_INCREF(lookup);
    d->cache = cache;
    d->lookup = lookup;
    d->vectorcall = dispatch_call;
    return reinterpret_cast<PyObject*>(d);
}

PyMethodDef g_methods[] = {
    {"call", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(call)), METH_FASTCALL,
     "call(name, *args): an entry point of the library; a non-zero status raises HipError"},
    {"set_hooks", set_hooks, METH_VARARGS, "set_hooks(general, failed)"},
    {"bind", bind, METH_O, "bind({name: (address, signature)}) -> number left out"},
    {"dispatcher", dispatcher, METH_VARARGS, "dispatcher(cache, lookup) -> dispatch"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_binding", "Calls into libminit_hip.so without ctypes.", -1, g_methods};

}  // namespace

PyMODINIT_FUNC PyInit__binding(void) {
    g_dispatcher_type.tp_name = "minit_amd._binding.dispatcher";
    g_dispatcher_type.tp_basicsize = sizeof(Dispatcher);
    g_dispatcher_type.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL;
    g_dispatcher_type.tp_vectorcall_offset = offsetof(Dispatcher, vectorcall);
    g_dispatcher_type.tp_call = PyVectorcall_Call;
    g_dispatcher_type.tp_dealloc = dispatcher_dealloc;
    if (PyType_Ready(&g_dispatcher_type) < 0) return nullptr;
    g_type_name = PyUnicode_InternFromString("type");
    if (g_type_name == nullptr) return nullptr;
    return PyModule_Create(&g_module);
}
