// The way from Python into the C ABI of include/bz_hip.h for the calls a step is made of.
//
// A launch costs 2.1 us on the host.  Through ctypes the call around it cost 1.5 us (rms_norm) to 3.5 us (decode_step, sixteen
// arguments and a table of fifteen fields), which is what small batches are bound by.  Here an argument that is what it usually
// is -- a tensor, an int, a float, None, a PageTable -- is converted in place; anything else (a subclass, a numpy scalar, a
// ctypes object) sends the whole call to the Python function it was bound with, which converts and refuses as ctypes does.
// Measured back to back: decode_step 9.0 -> 6.0 us, rms_norm 4.25 -> 2.9, the three calls at the ends of a step 12.5 -> 8.6.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <pthread.h>
#include <structmember.h>

#include <cstdint>
#include <cstring>
#include <utility>

#include "../../include/bz_hip.h"

namespace {

constexpr int kMaxArgs = 20;
union Slot {
    uint64_t u;
    float f;
};

template <class T> T slot_as(const Slot& s) {
    if constexpr (std::is_same<T, float>::value) return s.f;
    else if constexpr (std::is_pointer<T>::value) return reinterpret_cast<T>((uintptr_t)s.u);
    else return (T)s.u;
}
template <class F> struct Invoke;
template <class... A> struct Invoke<int(A...)> {
    static constexpr int kArgs = sizeof...(A);
    template <size_t... I> static int with(void* fn, const Slot* s, std::index_sequence<I...>) {
        return reinterpret_cast<int (*)(A...)>(fn)(slot_as<A>(s[I])...);
    }
    static int run(void* fn, const Slot* s) { return with(fn, s, std::index_sequence_for<A...>{}); }
};

// One letter per C argument: p address (tensor, int or None), d type code of a tensor, k PageTable, u unsigned, i int,
// t truth value as int, f float, s stream (None: torch's current one).
struct Entry {
    const char *name, *spec;
    int args;
    int (*run)(void*, const Slot*);
};
#define BZ_ENTRY(fn, spec) {#fn, spec, Invoke<decltype(fn)>::kArgs, Invoke<decltype(fn)>::run}
const Entry kEntries[] = {
    BZ_ENTRY(bz_batch_decode, "ppdkpduiffppps"),
    BZ_ENTRY(bz_batch_decode_noalloc, "ppdkpduiffppps"),
    BZ_ENTRY(bz_decode_step, "ppdppkpdutffppps"),
    BZ_ENTRY(bz_batch_prefill_ragged, "pppppppduuuutiffs"),
    BZ_ENTRY(bz_store_prefill_kv, "kppdpuputfpps"),
    BZ_ENTRY(bz_append_decode_kv, "kppdputfpps"),
    BZ_ENTRY(bz_rms_norm, "pppduufs"),
    BZ_ENTRY(bz_add_rms_norm, "pppduufs"),
    BZ_ENTRY(bz_silu_and_mul, "ppduus"),
    BZ_ENTRY(bz_add_residual, "ppduus"),
    BZ_ENTRY(bz_embedding, "ppppduus"),
    BZ_ENTRY(bz_gather_last_token, "pppduuus"),
    BZ_ENTRY(bz_batch_find_max, "ppduus"),
};

// What setup() was given: objects of torch and of the Python side that are looked at in every call.
PyObject *g_tensor, *g_data_ptr, *g_dtypes, *g_table, *g_initialized, *g_device, *g_raw_stream;
bool g_gpu_up; // torch has initialised the GPU in this process (a forked child asks again)
PyObject *s_dtype, *s_k_data, *s_v_data, *s_indices_d, *s_indptr_d, *s_last_page_len_d, *s_batch_size, *s_page_size, *s_num_heads,
    *s_head_size, *s_stride_page, *s_stride_n, *s_stride_h, *s_kv_dtype, *s_steps_ahead_d;

// Conversions: 1 done, 0 not one of the usual objects (the slow way decides), -1 an exception is set.
int address_of(PyObject* o, uint64_t& to) {
    if (o == Py_None) { to = 0; return 1; }
    if ((PyObject*)Py_TYPE(o) == g_tensor) {
        PyObject* v = PyObject_CallOneArg(g_data_ptr, o);
        if (!v) return -1;
        to = PyLong_AsUnsignedLongLongMask(v);
        Py_DECREF(v);
        return to == (uint64_t)-1 && PyErr_Occurred() ? -1 : 1;
    }
    if (!PyLong_CheckExact(o)) return 0;
    to = PyLong_AsUnsignedLongLongMask(o);
    return to == (uint64_t)-1 && PyErr_Occurred() ? -1 : 1;
}
int whole_of(PyObject* o, uint64_t& to) {
    if (!PyLong_CheckExact(o) && !PyBool_Check(o)) return 0;
    to = PyLong_AsUnsignedLongLongMask(o);
    return to == (uint64_t)-1 && PyErr_Occurred() ? -1 : 1;
}
int type_of(PyObject* o, uint64_t& to) {
    if ((PyObject*)Py_TYPE(o) != g_tensor) return 0;
    PyObject* t = PyObject_GetAttr(o, s_dtype);
    if (!t) return -1;
    PyObject* code = PyDict_GetItemWithError(g_dtypes, t); // (borrowed)
    Py_DECREF(t);
    if (!code) return PyErr_Occurred() ? -1 : 0;
    return whole_of(code, to);
}
int stream_of(PyObject* o, uint64_t& to) {
    if (o != Py_None) return PyLong_CheckExact(o) ? address_of(o, to) : 0;
    if (!g_gpu_up) {
        PyObject* up = PyObject_CallNoArgs(g_initialized);
        if (!up) return -1;
        const int yes = PyObject_IsTrue(up);
        Py_DECREF(up);
        if (yes <= 0) return yes;
        g_gpu_up = true;
    }
    PyObject* dev = PyObject_CallNoArgs(g_device);
    if (!dev) return -1;
    PyObject* v = PyObject_CallOneArg(g_raw_stream, dev);
    Py_DECREF(dev);
    if (!v) return -1;
    to = PyLong_AsUnsignedLongLongMask(v);
    Py_DECREF(v);
    return to == (uint64_t)-1 && PyErr_Occurred() ? -1 : 1;
}
int table_of(PyObject* o, bz_paged_kv_t& kv) {
    if ((PyObject*)Py_TYPE(o) != g_table) return 0;
    PyObject* d = PyObject_GenericGetDict(o, nullptr);
    if (!d) return -1;
    int rc = 1;
    auto get = [&](PyObject* name, int (*convert)(PyObject*, uint64_t&)) -> uint64_t {
        if (rc != 1) return 0;
        PyObject* v = PyDict_GetItemWithError(d, name);
        uint64_t to = 0;
        if (!v) { rc = PyErr_Occurred() ? -1 : 0; return 0; }
        Py_INCREF(v);
        rc = convert(v, to);
        Py_DECREF(v);
        return to;
    };
    kv = bz_paged_kv_t{};
    kv.k_data = (void*)get(s_k_data, address_of);
    kv.v_data = (void*)get(s_v_data, address_of);
    kv.indices = (const int32_t*)get(s_indices_d, address_of);
    kv.indptr = (const int32_t*)get(s_indptr_d, address_of);
    kv.last_page_len = (const int32_t*)get(s_last_page_len_d, address_of);
    kv.batch_size = (uint32_t)get(s_batch_size, whole_of);
    kv.page_size = (uint32_t)get(s_page_size, whole_of);
    kv.num_kv_heads = (uint32_t)get(s_num_heads, whole_of);
    kv.head_dim = (uint32_t)get(s_head_size, whole_of);
    kv.stride_page = get(s_stride_page, whole_of);
    kv.stride_n = get(s_stride_n, whole_of);
    kv.stride_h = get(s_stride_h, whole_of);
    kv.kv_dtype = (int)get(s_kv_dtype, whole_of);
    kv.steps_ahead = (const int32_t*)get(s_steps_ahead_d, address_of);
    Py_DECREF(d);
    return rc;
}

struct Call {
    PyObject_HEAD
    vectorcallfunc vectorcall;
    const Entry* entry;
    void* fn;
    PyObject *slow, *check, *what;
};

PyObject* call(PyObject* self_, PyObject* const* args, size_t nargsf, PyObject* kwnames) {
    Call* self = (Call*)self_;
    const Entry& e = *self->entry;
    if (PyVectorcall_NARGS(nargsf) != e.args || (kwnames && PyTuple_GET_SIZE(kwnames))) {
        PyErr_Format(PyExc_TypeError, "%s takes %d positional arguments", e.name, e.args);
        return nullptr;
    }
    Slot slot[kMaxArgs];
    bz_paged_kv_t kv;
    int rc = 1;
    for (int i = 0; i < e.args && rc == 1; ++i) {
        PyObject* o = args[i];
        uint64_t u = 0;
        switch (e.spec[i]) {
            case 'p': rc = address_of(o, u); break;
            case 'd': rc = type_of(o, u); break;
            case 's': rc = stream_of(o, u); break;
            case 'k': rc = table_of(o, kv); u = (uint64_t)(uintptr_t)&kv; break;
            case 'f':
                if (PyFloat_CheckExact(o)) { slot[i].f = (float)PyFloat_AS_DOUBLE(o); continue; }
                rc = 0;
                break;
            default: rc = whole_of(o, u); break;
        }
        slot[i].u = u;
    }
    if (rc < 0) return nullptr;
    PyObject* code;
    if (rc == 0) {
        code = PyObject_Vectorcall(self->slow, args, (size_t)e.args, nullptr);
        if (!code) return nullptr;
    } else {
        int result;
        Py_BEGIN_ALLOW_THREADS
        result = e.run(self->fn, slot);
        Py_END_ALLOW_THREADS
        if (result == 0) Py_RETURN_NONE;
        code = PyLong_FromLong(result);
        if (!code) return nullptr;
    }
    PyObject* done = PyObject_CallFunctionObjArgs(self->check, code, self->what, nullptr); // raises for every code but 0
    Py_DECREF(code);
    return done;
}

void call_free(PyObject* self_) {
    Call* self = (Call*)self_;
    Py_XDECREF(self->slow);
    Py_XDECREF(self->check);
    Py_XDECREF(self->what);
    PyTypeObject* type = Py_TYPE(self_);
    type->tp_free(self_);
    Py_DECREF(type); // (an instance of a heap type holds it)
}

PyMemberDef call_members[] = {{"__vectorcalloffset__", T_PYSSIZET, offsetof(Call, vectorcall), READONLY, nullptr}, {nullptr}};
PyType_Slot call_slots[] = {{Py_tp_dealloc, (void*)call_free}, {Py_tp_call, (void*)PyVectorcall_Call}, {Py_tp_members, call_members}, {0, nullptr}};
PyType_Spec call_spec = {"bz_pycall.Call", sizeof(Call), 0, Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL, call_slots};
PyTypeObject* g_call_type;

// bind(name, address, slow, check, what): the call of that name at that address
PyObject* bind(PyObject*, PyObject* args) {
    const char* name;
    unsigned long long address;
    PyObject *slow, *check, *what;
    if (!PyArg_ParseTuple(args, "sKOOO", &name, &address, &slow, &check, &what)) return nullptr;
    for (const Entry& e : kEntries) {
        if (strcmp(e.name, name)) continue;
        Call* c = (Call*)g_call_type->tp_alloc(g_call_type, 0);
        if (!c) return nullptr;
        c->vectorcall = call;
        c->entry = &e;
        c->fn = (void*)(uintptr_t)address;
        Py_INCREF(slow); Py_INCREF(check); Py_INCREF(what);
        c->slow = slow; c->check = check; c->what = what;
        return (PyObject*)c;
    }
    return PyErr_Format(PyExc_KeyError, "no call of the name %s", name);
}

// setup(tensor type, its data_ptr, type codes by dtype, PageTable, is_initialized, current device, raw stream of a device)
PyObject* setup(PyObject*, PyObject* args) {
    PyObject* o[7];
    if (!PyArg_ParseTuple(args, "OOO!OOOO", &o[0], &o[1], &PyDict_Type, &o[2], &o[3], &o[4], &o[5], &o[6])) return nullptr;
    PyObject** to[7] = {&g_tensor, &g_data_ptr, &g_dtypes, &g_table, &g_initialized, &g_device, &g_raw_stream};
    for (int i = 0; i < 7; ++i) {
        Py_INCREF(o[i]);
        Py_XSETREF(*to[i], o[i]);
    }
    g_gpu_up = false; // (as the function before this one saw it)
    Py_RETURN_NONE;
}

PyObject* specs(PyObject*, PyObject*) { // {name: spec}
    PyObject* d = PyDict_New();
    for (const Entry& e : kEntries) {
        PyObject* s = d ? PyUnicode_FromString(e.spec) : nullptr;
        if (!s || PyDict_SetItemString(d, e.name, s)) { Py_XDECREF(s); Py_XDECREF(d); return nullptr; }
        Py_DECREF(s);
    }
    return d;
}

PyMethodDef methods[] = {{"bind", bind, METH_VARARGS, nullptr}, {"setup", setup, METH_VARARGS, nullptr}, {"specs", specs, METH_NOARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "bz_pycall", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

} // namespace

PyMODINIT_FUNC PyInit_bz_pycall() {
    for (const Entry& e : kEntries)
        if ((int)strlen(e.spec) != e.args || e.args > kMaxArgs)
            return PyErr_Format(PyExc_SystemError, "%s has %d arguments", e.name, e.args);
    const struct { PyObject** to; const char* name; } names[] = {
        {&s_dtype, "dtype"}, {&s_k_data, "k_data"}, {&s_v_data, "v_data"}, {&s_indices_d, "indices_d"}, {&s_indptr_d, "indptr_d"},
        {&s_last_page_len_d, "last_page_len_d"}, {&s_batch_size, "batch_size"}, {&s_page_size, "page_size"}, {&s_num_heads, "num_heads"},
        {&s_head_size, "head_size"}, {&s_stride_page, "stride_page"}, {&s_stride_n, "stride_n"}, {&s_stride_h, "stride_h"},
        {&s_kv_dtype, "kv_dtype"}, {&s_steps_ahead_d, "steps_ahead_d"}};
    for (const auto& n : names)
        if (!(*n.to = PyUnicode_InternFromString(n.name))) return nullptr;
    if (!(g_call_type = (PyTypeObject*)PyType_FromSpec(&call_spec))) return nullptr;
    pthread_atfork(nullptr, nullptr, [] { g_gpu_up = false; });
    return PyModule_Create(&module);
}
