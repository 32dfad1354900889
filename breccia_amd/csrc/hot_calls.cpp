// The entry points that a serving loop calls for every layer, as a CPython module of their own (breccia_amd._hot).
//
// What bounds such a call is the host: a kernel launch costs 2.7 to 4 us of it, the kernels of a short step 6 and 2 us
// of the device, and a call through ctypes with arrays turned into pointers one by one another 2 to 4 us.  Here the
// arguments are read straight out of the Python objects (0.2 us).
//
// Only plain arguments are taken: int and float objects that fit, None or an int (or c_void_p, or the owning class)
// for an address, C-contiguous native int32 / int64 numpy arrays of equal sizes.  For anything else the functions
// return NotImplemented, having done nothing, and kv.py makes the call as it always could, with ctypes' conversions and
// its own errors.  Otherwise they return the library's status (seq_reserve: the list of pairs on success).  The
// library is called without the GIL, as ctypes does.
//
// The module is not linked against the library: kv.py hands it the entry points of the one that ctypes has loaded
// (bind).  A dependency is looked for along LD_LIBRARY_PATH first, and with another copy of the library there, pools
// made by one were read by the other.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#define NPY_NO_DEPRECATED_API NPY_1_7_API_VERSION
#include <numpy/arrayobject.h>

#include <cstdint>
#include <type_traits>

#include "../../include/breccia_kv.h"

namespace {

PyObject* g_c_void_p = nullptr;  // ctypes.c_void_p
PyObject* g_buffer = nullptr;    // kv.DeviceBuffer, its address in .ptr
PyObject* g_stream = nullptr;    // kv.Stream, its address in .handle
PyObject* g_ptr_name = nullptr;
PyObject* g_handle_name = nullptr;

// The library's entry points; null until bind().
#define ENTRY_POINTS(X) \
    X(bkv_append) X(bkv_append_f16) X(bkv_append_kprep) X(bkv_decode_attn) X(bkv_decode_step) X(bkv_decode_attn_select) \
    X(bkv_prefill_attn) X(bkv_idx_pool) X(bkv_select_blocks) X(bkv_seq_reserve)
#define POINTER(name) decltype(&::name) name = nullptr;
struct Library {
    ENTRY_POINTS(POINTER)
};
#undef POINTER
Library g_lib;
bool g_bound = false;

// Reads the positional arguments of one call in turn; `ok` falls, and stays down, at the first that is not plain.
class Reader {
   public:
    Reader(PyObject* const* args, Py_ssize_t n, Py_ssize_t want) : at_(args), ok(n == want && g_bound) {}

    int32_t i32() {
        const int64_t v = i64();
        if (v < INT32_MIN || v > INT32_MAX) ok = false;
        return (int32_t)v;
    }
    int64_t i64() {
        PyObject* o = next();
        if (!ok || !PyLong_CheckExact(o)) return ok = false, 0;
        int over = 0;
        const long long v = PyLong_AsLongLongAndOverflow(o, &over);
        if (over) ok = false;
        return v;
    }
    float f32() {
        PyObject* o = next();
        if (!ok || !PyFloat_CheckExact(o)) return ok = false, 0.0f;
        return (float)PyFloat_AS_DOUBLE(o);
    }
    bool flag() {
        PyObject* o = next();
        if (!ok || !PyBool_Check(o)) return ok = false, false;
        return o == Py_True;
    }
    template <typename T = void>
    T* device() {
        return static_cast<T*>(address(next(), g_buffer, g_ptr_name));
    }
    void* stream() { return address(next(), g_stream, g_handle_name); }
    bkv_pool* pool() { return static_cast<bkv_pool*>(address(next(), nullptr, nullptr)); }
    const int32_t* i32s(Py_ssize_t& n) { return static_cast<const int32_t*>(array(n, NPY_INT32)); }
    const int64_t* i64s(Py_ssize_t& n) { return static_cast<const int64_t*>(array(n, NPY_INT64)); }
    // a list of device addresses, at most `cap` of them
    void device_list(const float** out, Py_ssize_t cap, Py_ssize_t& n) {
        PyObject* o = next();
        n = 0;
        if (!ok || !PyList_CheckExact(o) || PyList_GET_SIZE(o) > cap) return (void)(ok = false);
        n = PyList_GET_SIZE(o);
        // the length is looked at again: reading an owner's attribute may run Python code
        for (Py_ssize_t i = 0; ok && i < n; ++i) {
            if (PyList_GET_SIZE(o) != n) return (void)(ok = false);
            PyObject* item = PyList_GET_ITEM(o, i);
            Py_INCREF(item);
            out[i] = static_cast<const float*>(address(item, g_buffer, g_ptr_name));
            Py_DECREF(item);
        }
    }

   private:
    PyObject* const* at_;

   public:
    bool ok;

   private:
    PyObject* next() { return ok ? *at_++ : nullptr; }

    const void* array(Py_ssize_t& n, int type) {
        PyObject* o = next();
        n = 0;
        if (!ok || !PyArray_CheckExact(o)) return ok = false, nullptr;
        PyArrayObject* a = reinterpret_cast<PyArrayObject*>(o);
        if (PyArray_TYPE(a) != type || !PyArray_ISCARRAY_RO(a)) return ok = false, nullptr;
        n = PyArray_SIZE(a);
        return PyArray_DATA(a);
    }
    void* address(PyObject* o, PyObject* owner, PyObject* member) {
        if (!ok) return nullptr;
        if (o == Py_None) return nullptr;
        if (PyLong_CheckExact(o)) {
            int over = 0;
            const long long v = PyLong_AsLongLongAndOverflow(o, &over);
            if (over || v < 0) ok = false;
            return reinterpret_cast<void*>(static_cast<uintptr_t>(v));
        }
        if (reinterpret_cast<PyObject*>(Py_TYPE(o)) == g_c_void_p) return held(o);
        if (owner && reinterpret_cast<PyObject*>(Py_TYPE(o)) == owner) {
            PyObject* p = PyObject_GetAttr(o, member);
            void* v = p ? address(p, nullptr, nullptr) : nullptr;
            if (!p) PyErr_Clear(), ok = false;
            Py_XDECREF(p);
            return v;
        }
        ok = false;
        return nullptr;
    }
    // what a c_void_p object holds
    void* held(PyObject* o) {
        Py_buffer view;
        if (PyObject_GetBuffer(o, &view, PyBUF_SIMPLE) != 0) {
            PyErr_Clear();
            return ok = false, nullptr;
        }
        void* v = nullptr;
        if (view.len == (Py_ssize_t)sizeof v) v = *static_cast<void**>(view.buf);
        else ok = false;
        PyBuffer_Release(&view);
        return v;
    }
};

PyObject* not_plain() { Py_RETURN_NOTIMPLEMENTED; }

// the library's status, from a call made without the GIL
template <typename Call>
PyObject* status_of(Call call) {
    bkv_status st;
    Py_BEGIN_ALLOW_THREADS;
    st = call();
    Py_END_ALLOW_THREADS;
    return PyLong_FromLong((long)st);
}

PyObject* append(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    Reader r(args, n_args, 9);
    bkv_pool* pool = r.pool();
    const int32_t layer = r.i32();
    Py_ssize_t n, n1, n2;
    const int32_t* seqs = r.i32s(n);
    const int64_t* pos0 = r.i64s(n1);
    const int32_t* n_tokens = r.i32s(n2);
    const void *k = r.device(), *v = r.device();
    void* stream = r.stream();
    const bool f16_rows = r.flag();
    if (!r.ok || n != n1 || n != n2 || n > INT32_MAX) return not_plain();
    return status_of([&] {
        return f16_rows ? g_lib.bkv_append_f16(pool, layer, (int32_t)n, seqs, pos0, n_tokens, static_cast<const uint16_t*>(k),
                                         static_cast<const uint16_t*>(v), stream)
                        : g_lib.bkv_append(pool, layer, (int32_t)n, seqs, pos0, n_tokens, static_cast<const float*>(k),
                                     static_cast<const float*>(v), stream);
    });
}

PyObject* append_kprep(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    Reader r(args, n_args, 14);
    bkv_pool* pool = r.pool();
    const int32_t layer = r.i32();
    Py_ssize_t n, n1, n2;
    const int32_t* seqs = r.i32s(n);
    const int64_t* pos0 = r.i64s(n1);
    const int32_t* n_tokens = r.i32s(n2);
    const float *k = r.device<float>(), *v = r.device<float>(), *gamma = r.device<float>();
    const float eps = r.f32();
    const float* table = r.device<float>();
    const int32_t n_rot = r.i32(), max_pos = r.i32();
    const int32_t* positions = r.device<int32_t>();
    void* stream = r.stream();
    if (!r.ok || n != n1 || n != n2 || n > INT32_MAX) return not_plain();
    return status_of([&] {
        return g_lib.bkv_append_kprep(pool, layer, (int32_t)n, seqs, pos0, n_tokens, k, v, gamma, eps, table, n_rot, max_pos, positions,
                                stream);
    });
}

PyObject* decode_attn(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    Reader r(args, n_args, 12);
    bkv_pool* pool = r.pool();
    const int32_t layer = r.i32();
    Py_ssize_t n, n1;
    const int32_t* seqs = r.i32s(n);
    const int64_t* pos = r.i64s(n1);
    const int32_t n_q = r.i32();
    const float* q = r.device<float>();
    float* out = r.device<float>();
    const float scale = r.f32();
    const float* gate = r.device<float>();
    const int64_t seq_stride = r.i64(), head_stride = r.i64();
    void* stream = r.stream();
    if (!r.ok || n != n1 || n > INT32_MAX) return not_plain();
    return status_of([&] {
        return g_lib.bkv_decode_attn(pool, layer, (int32_t)n, seqs, pos, n_q, q, gate, seq_stride, head_stride, scale, out, stream);
    });
}

PyObject* decode_step(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    Reader r(args, n_args, 14);
    bkv_pool* pool = r.pool();
    const int32_t layer = r.i32();
    Py_ssize_t n, n1;
    const int32_t* seqs = r.i32s(n);
    const int64_t* pos = r.i64s(n1);
    const float *k = r.device<float>(), *v = r.device<float>();
    const int32_t n_q = r.i32();
    const float* q = r.device<float>();
    float* out = r.device<float>();
    const float scale = r.f32();
    const float* gate = r.device<float>();
    const int64_t seq_stride = r.i64(), head_stride = r.i64();
    void* stream = r.stream();
    if (!r.ok || n != n1 || n > INT32_MAX) return not_plain();
    return status_of([&] {
        return g_lib.bkv_decode_step(pool, layer, (int32_t)n, seqs, pos, k, v, n_q, q, gate, seq_stride, head_stride, scale, out, stream);
    });
}

PyObject* decode_attn_select(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    Reader r(args, n_args, 16);
    bkv_pool* pool = r.pool();
    const int32_t layer = r.i32();
    Py_ssize_t n, n1;
    const int32_t* seqs = r.i32s(n);
    const int64_t* pos = r.i64s(n1);
    const int32_t n_q = r.i32();
    const float* q = r.device<float>();
    float* out = r.device<float>();
    const float scale = r.f32();
    const uint32_t* ids = r.device<uint32_t>();
    const int64_t id_stride = r.i64();
    const uint32_t* counts = r.device<uint32_t>();
    const int32_t max_ids = r.i32();
    const float* gate = r.device<float>();
    const int64_t seq_stride = r.i64(), head_stride = r.i64();
    void* stream = r.stream();
    if (!r.ok || n != n1 || n > INT32_MAX) return not_plain();
    return status_of([&] {
        return g_lib.bkv_decode_attn_select(pool, layer, (int32_t)n, seqs, pos, n_q, q, gate, seq_stride, head_stride, scale, ids, id_stride,
                                      counts, max_ids, out, stream);
    });
}

PyObject* prefill_attn(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    Reader r(args, n_args, 13);
    bkv_pool* pool = r.pool();
    const int32_t layer = r.i32();
    Py_ssize_t n, n1, n2;
    const int32_t* seqs = r.i32s(n);
    const int64_t* pos0 = r.i64s(n1);
    const int32_t* n_tokens = r.i32s(n2);
    const int32_t n_q = r.i32();
    const float* q = r.device<float>();
    float* out = r.device<float>();
    const float scale = r.f32();
    const float* gate = r.device<float>();
    const int64_t tok_stride = r.i64(), head_stride = r.i64();
    void* stream = r.stream();
    if (!r.ok || n != n1 || n != n2 || n > INT32_MAX) return not_plain();
    return status_of([&] {
        return g_lib.bkv_prefill_attn(pool, layer, (int32_t)n, seqs, pos0, n_tokens, n_q, q, gate, tok_stride, head_stride, scale, out, stream);
    });
}

PyObject* idx_pool(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    Reader r(args, n_args, 14);
    bkv_pool* pool = r.pool();
    float* pooled = r.device<float>();
    const int32_t max_blocks = r.i32();
    float* tail = r.device<float>();
    const float* idx_k = r.device<float>();
    const int64_t pos0 = r.i64();
    const int32_t tokens = r.i32();
    const float* gamma = r.device<float>();
    const float eps = r.f32();
    const float* table = r.device<float>();
    const int32_t n_rot = r.i32(), max_pos = r.i32(), idx_dim = r.i32();
    void* stream = r.stream();
    if (!r.ok) return not_plain();
    return status_of([&] {
        return g_lib.bkv_idx_pool(pool, pooled, max_blocks, tail, idx_k, pos0, tokens, gamma, eps, table, n_rot, max_pos, idx_dim, stream);
    });
}

PyObject* select_blocks(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    Reader r(args, n_args, 13);
    bkv_pool* pool = r.pool();
    Py_ssize_t n, n1, n2;
    const int64_t* pos = r.i64s(n);
    const float* idx_q = r.device<float>();
    const float* pooled[BKV_MAX_BATCH];
    r.device_list(pooled, BKV_MAX_BATCH, n1);
    const int32_t* n_blocks = r.i32s(n2);
    const int32_t n_head = r.i32(), idx_dim = r.i32(), topk = r.i32();
    uint32_t* ids = r.device<uint32_t>();
    const int64_t id_stride = r.i64();
    uint32_t* counts = r.device<uint32_t>();
    const int32_t max_ids = r.i32();
    void* stream = r.stream();
    if (!r.ok || n != n1 || n != n2) return not_plain();
    return status_of([&] {
        return g_lib.bkv_select_blocks(pool, (int32_t)n, pos, idx_q, pooled, n_blocks, n_head, idx_dim, topk, ids, id_stride, counts, max_ids,
                                 stream);
    });
}

PyObject* seq_reserve(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    constexpr int32_t kPairs = 64;
    Reader r(args, n_args, 4);
    bkv_pool* pool = r.pool();
    const int32_t seq = r.i32();
    const int64_t new_len = r.i64();
    const int32_t capacity = r.i32();
    if (!r.ok || capacity < 1 || capacity > kPairs) return not_plain();
    bkv_page_pair pairs[kPairs];
    int32_t n = 0;
    bkv_status st;
    Py_BEGIN_ALLOW_THREADS;
    st = g_lib.bkv_seq_reserve(pool, seq, new_len, pairs, capacity, &n);
    Py_END_ALLOW_THREADS;
    if (st != BKV_OK) return PyLong_FromLong((long)st);
    PyObject* list = PyList_New(n);
    for (int32_t i = 0; list && i < n; ++i) {
        PyObject* pair = Py_BuildValue("(ii)", (int)pairs[i].src, (int)pairs[i].dst);
        if (!pair) {
            Py_DECREF(list);
            return nullptr;
        }
        PyList_SET_ITEM(list, i, pair);
    }
    return list;
}

// bind(c_void_p, DeviceBuffer, Stream, {name: address}): the classes whose objects are read as addresses, and the
// library's entry points
PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
    if (n_args != 4 || !PyDict_Check(args[3])) {
        PyErr_SetString(PyExc_TypeError, "bind takes three classes and the entry points' addresses");
        return nullptr;
    }
    Library found;
    const auto take = [&](const char* name, auto& entry) {
        PyObject* at = PyDict_GetItemString(args[3], name);
        void* p = at ? PyLong_AsVoidPtr(at) : nullptr;
        if (!p && !PyErr_Occurred()) PyErr_Format(PyExc_ValueError, "no address of %s", name);
        entry = reinterpret_cast<std::remove_reference_t<decltype(entry)>>(p);
        return p != nullptr;
    };
#define TAKE(name) \
    if (!take(#name, found.name)) return nullptr;
    ENTRY_POINTS(TAKE)
#undef TAKE
    PyObject** const kept[3] = {&g_c_void_p, &g_buffer, &g_stream};
    for (int i = 0; i < 3; ++i) {
        Py_INCREF(args[i]);
        Py_XSETREF(*kept[i], args[i]);
    }
    g_lib = found;
    g_bound = true;
    Py_RETURN_NONE;
}

#define HOT_CALL(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(name)), METH_FASTCALL, nullptr}
PyMethodDef g_methods[] = {HOT_CALL(append),
                           HOT_CALL(append_kprep),
                           HOT_CALL(decode_attn),
                           HOT_CALL(decode_step),
                           HOT_CALL(decode_attn_select),
                           HOT_CALL(prefill_attn),
                           HOT_CALL(idx_pool),
                           HOT_CALL(select_blocks),
                           HOT_CALL(seq_reserve),
                           HOT_CALL(bind),
                           {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_hot", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__hot(void) {
    import_array();
    g_ptr_name = PyUnicode_InternFromString("ptr");
    g_handle_name = PyUnicode_InternFromString("handle");
    if (!g_ptr_name || !g_handle_name) return nullptr;
    return PyModule_Create(&g_module);
}
