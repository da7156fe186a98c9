// What a launch costs the host beside the launch itself: the binding's four small functions (_lib.py: call, require_gpu, ptr, stream) as a CPython extension.  A served step of one token
// or a training step on a few rows is hundreds of launches of a few microseconds; ctypes converted their 10 to 35 arguments, and Python looked the stream up, in 6 us of each
// launch's 17 (the launch itself: 3).  The semantics are _lib.py's own, and everything out of the ordinary -- an argument that is no int / float / None, a wrong count, operands
// that are no HIP tensors, a device other than the current one, a library that is not loaded yet -- goes to the Python functions that stand there.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <string.h>

#include <tuple>
#include <type_traits>
#include <utility>

#include "../../include/mi355_vlm.h"

#define MI355_ENTRIES(E) \
    E(gemm_bf16) E(gemm_bf16_grouped) E(gemm_bf16_grouped_ws) E(gemm_bf16_attn_delta) E(adamw) E(colsum) E(rmsnorm_fwd) E(rmsnorm_bwd) E(reduce_rows_f32) E(qknorm_rope_fwd) E(qknorm_rope_bwd) \
    E(swiglu_fwd) E(swiglu_bwd) E(attn_fwd) E(attn_bwd) E(attn_bwd_ws) E(attn_bwd_qnorm) E(cross_entropy) E(ce_finalize) E(embedding_fwd) E(embedding_bwd) \
    E(embedding_bwd_sorted) E(copy2d) E(transpose_bf16) E(patchify) E(layernorm_fwd) E(layernorm_bwd_bf16) E(reduce_rows_into) E(reduce_rows_each) E(layernorm_bwd) E(cast) \
    E(vit_embed_assemble) E(split3_bf16) E(attn_f32_fwd) E(sumsq) E(clip_scale) E(add_f32_to_bf16) E(scale_bf16) E(gelu_fwd) E(gelu_bwd) E(gelu_bwd_colsum) E(patchify3d) \
    E(merge_patches) E(scatter_rows) E(zc_weight) E(mrope_table) E(rowmask) E(headnorm_rope_fwd) E(headnorm_rope_bwd) E(sigmoid_gate_fwd) E(sigmoid_gate_bwd) \
    E(attn_generic_fwd) E(attn_generic_bwd) E(gdn_gates_fwd) E(gdn_gates_bwd) E(causal_conv_silu_fwd) E(causal_conv_silu_bwd) E(l2norm_fwd) E(l2norm_bwd) \
    E(gated_delta_rule_fwd) E(causal_conv_silu_step) E(gated_delta_rule_bwd) E(gdr_chunked_fwd) E(gdr_chunked_bwd) E(gated_rmsnorm_fwd) E(gated_rmsnorm_bwd) \
    E(resize_h_u8) E(resize_v_normalize) E(pad_tokens) E(gemv_bf16) E(gemv_bf16_f32out) E(gemv_bf16_pro) E(decode_block) E(decode_blocks) E(attn_decode_qkv) E(decode_advance) \
    E(attn_decode) E(kv_append_rows) E(kv_append) E(argmax_rows) E(argmax_rows_f32) E(embed_hash_fwd) E(add_layernorm_fwd) E(rmsnorm_rows) E(delta_rule_tokens) \
    E(delta_chunked) E(latent_kv_append) E(rope_heads) E(gated_headnorm) E(gla_fwd) E(gla_fwd_below) E(router_logits) E(moe_route) E(moe_dispatch) E(moe_choose) E(moe_table_dispatch) \
    E(bgemm) E(latent_attn) E(group_rmsnorm_sum) E(ragged_conv) E(qkv_rows_append) E(delta_rule_ragged) E(glu_rows) E(sandwich_rmsnorm) E(pool_rows_update) E(act_rows) \
    E(dyt_sum) E(token_shift) E(linrec_ragged) E(rglru_ragged) E(gated_groupnorm) E(unary_rows) E(mingru_ragged) E(depth_sum) E(diff_attn) E(diff_join) E(hyper_mix) \
    E(mfma_pipe_probe) E(rope_apply) E(dropout) E(attn_dropout_fwd) E(attn_generic_dropout_fwd) E(attn_generic_dropout_bwd) E(attn_dropout_bwd)

namespace {

thread_local int tls_device = -1;  // index of the device of the operands that this THREAD's last require_gpu() saw; -1: none

PyObject *s_is_cuda, *s_get_device, *s_data_ptr;     // interned names
PyObject *fn_device, *fn_stream;                     // torch._C._cuda_getDevice, torch._C._cuda_getCurrentRawStream
PyObject *slow_call, *slow_require, *slow_fail;      // _lib.py's Python forms; slow_fail(name, rc) raises
PyObject* table;                                     // entry name -> its place in `entries`

// ---- arguments: false (and no exception) where the value is not of the kind that converts here
inline bool convert(PyObject* o, void*& out) {
    if (o == Py_None) return out = nullptr, true;
    if (!PyLong_Check(o)) return false;
    out = reinterpret_cast<void*>(PyLong_AsUnsignedLongLongMask(o));
    return true;
}
template <class T>
inline std::enable_if_t<std::is_pointer_v<T>, bool> convert(PyObject* o, T& out) {
    void* p;
    if (!convert(o, p)) return false;
    out = reinterpret_cast<T>(p);
    return true;
}
template <class T>
inline std::enable_if_t<std::is_integral_v<T>, bool> convert(PyObject* o, T& out) {  // masked to the width, as ctypes does
    if (!PyLong_Check(o)) return false;
    out = static_cast<T>(PyLong_AsUnsignedLongLongMask(o));
    return true;
}
inline bool convert(PyObject* o, float& out) {
    if (PyFloat_Check(o)) return out = static_cast<float>(PyFloat_AS_DOUBLE(o)), true;
    if (!PyLong_Check(o)) return false;
    const double d = PyLong_AsDouble(o);
    if (d == -1.0 && PyErr_Occurred()) return PyErr_Clear(), false;
    return out = static_cast<float>(d), true;
}

struct Entry {
    const char* name;
    int args;  // without the stream
    void* address;
    bool (*invoke)(void* address, PyObject* const* args, void* stream, int& rc);
};

template <class... A>
struct Invoke {
    static_assert(sizeof...(A) > 1, "an entry point has arguments and a stream");
    static constexpr int N = static_cast<int>(sizeof...(A)) - 1;
    template <size_t... I>
    static bool with(void* address, PyObject* const* args, void* stream, int& rc, std::index_sequence<I...>) {
        std::tuple<A...> v{};
        if (!(convert(args[I], std::get<I>(v)) && ...)) return false;
        std::get<N>(v) = stream;
        Py_BEGIN_ALLOW_THREADS
        rc = reinterpret_cast<int (*)(A...)>(address)(std::get<I>(v)..., std::get<N>(v));
        Py_END_ALLOW_THREADS
        return true;
    }
    static bool run(void* address, PyObject* const* args, void* stream, int& rc) { return with(address, args, stream, rc, std::make_index_sequence<N>{}); }
};
template <class... A>
constexpr Entry entry(const char* name, int (*)(A...)) {
    static_assert(std::is_same_v<std::tuple_element_t<sizeof...(A) - 1, std::tuple<A...>>, void*>, "the last argument is the stream");
    return Entry{name, Invoke<A...>::N, nullptr, &Invoke<A...>::run};
}
Entry entries[] = {
#define E(n) entry("mi355_" #n, static_cast<decltype(&mi355_##n)>(nullptr)),
    MI355_ENTRIES(E)
#undef E
};
constexpr int ENTRIES = static_cast<int>(sizeof(entries) / sizeof(entries[0]));

// raw handle of the current stream of device `index`; false: an exception is set
bool current_stream(int index, void*& stream) {
    PyObject* i = PyLong_FromLong(index);
    if (!i) return false;
    PyObject* h = PyObject_CallOneArg(fn_stream, i);
    Py_DECREF(i);
    if (!h) return false;
    stream = PyLong_AsVoidPtr(h);
    Py_DECREF(h);
    return !PyErr_Occurred();
}

PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n >= 1 && tls_device >= 0) {
        PyObject* at = PyDict_GetItemWithError(table, args[0]);
        if (!at && PyErr_Occurred()) return nullptr;
        Entry* e = at ? &entries[PyLong_AsLong(at)] : nullptr;
        if (e && e->address && n - 1 == e->args) {
            PyObject* cur = PyObject_CallNoArgs(fn_device);
            if (!cur) return nullptr;
            const long device = PyLong_AsLong(cur);
            Py_DECREF(cur);
            if (device == tls_device) {
                void* stream;
                int rc = 0;
                if (!current_stream(tls_device, stream)) return nullptr;
                if (e->invoke(e->address, args + 1, stream, rc)) {
                    if (rc == 0) Py_RETURN_NONE;
                    PyObject* code = PyLong_FromLong(rc);
                    if (!code) return nullptr;
                    PyObject* r = PyObject_CallFunctionObjArgs(slow_fail, args[0], code, nullptr);
                    Py_DECREF(code);
                    return r;
                }
            }
        }
    }
    return PyObject_Vectorcall(slow_call, args, static_cast<size_t>(n), nullptr);
}

PyObject* require_gpu(PyObject*, PyObject* const* args, Py_ssize_t n) {
    int device = -1;
    for (Py_ssize_t i = 0; i < n; ++i) {
        if (args[i] == Py_None) continue;
        PyObject* c = PyObject_GetAttr(args[i], s_is_cuda);
        if (!c) return nullptr;
        const bool cuda = c == Py_True;
        Py_DECREF(c);
        long index = -1;
        if (cuda) {
            PyObject* d = PyObject_CallMethodNoArgs(args[i], s_get_device);
            if (!d) return nullptr;
            index = PyLong_AsLong(d);
            Py_DECREF(d);
        }
        if (index < 0 || (device >= 0 && index != device)) {  // not ours to launch on: _lib.py says why
            return PyObject_Vectorcall(slow_require, args, static_cast<size_t>(n), nullptr);
        }
        device = static_cast<int>(index);
    }
    tls_device = device;
    Py_RETURN_NONE;
}

PyObject* ptr(PyObject*, PyObject* t) {
    if (t == Py_None) Py_RETURN_NONE;
    return PyObject_CallMethodNoArgs(t, s_data_ptr);
}

PyObject* bind(PyObject*, PyObject* args) {
    const char* name;
    unsigned long long address;
    if (!PyArg_ParseTuple(args, "sK", &name, &address)) return nullptr;
    for (Entry& e : entries)
        if (!strcmp(e.name, name)) {
            e.address = reinterpret_cast<void*>(address);
            Py_RETURN_TRUE;
        }
    Py_RETURN_FALSE;
}

PyObject* device(PyObject*, PyObject*) { return PyLong_FromLong(tls_device); }
PyObject* set_device(PyObject*, PyObject* o) {
    const long d = PyLong_AsLong(o);
    if (d == -1 && PyErr_Occurred()) return nullptr;
    tls_device = static_cast<int>(d);
    Py_RETURN_NONE;
}

PyObject* setup(PyObject*, PyObject* args) {  // (getDevice, getCurrentRawStream, call, require_gpu, fail)
    PyObject* f[5];
    if (!PyArg_ParseTuple(args, "OOOOO", &f[0], &f[1], &f[2], &f[3], &f[4])) return nullptr;
    PyObject** to[5] = {&fn_device, &fn_stream, &slow_call, &slow_require, &slow_fail};
    for (int i = 0; i < 5; ++i) {
        Py_INCREF(f[i]);
        Py_XSETREF(*to[i], f[i]);
    }
    Py_RETURN_NONE;
}

PyObject* names(PyObject*, PyObject*) {
    PyObject* l = PyList_New(ENTRIES);
    for (int i = 0; l && i < ENTRIES; ++i) PyList_SET_ITEM(l, i, PyUnicode_FromString(entries[i].name));
    return l;
}

PyMethodDef methods[] = {
    {"call", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(call)), METH_FASTCALL, "call(name, *args): _lib.call"},
    {"require_gpu", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(require_gpu)), METH_FASTCALL, "require_gpu(*tensors): _lib.require_gpu"},
    {"ptr", ptr, METH_O, "ptr(tensor or None): _lib.ptr"},
    {"bind", bind, METH_VARARGS, "bind(name, address): where an entry point of the loaded library is"},
    {"device", device, METH_NOARGS, "index of the device of this thread's last require_gpu, -1: none"},
    {"set_device", set_device, METH_O, "sets what device() gives"},
    {"setup", setup, METH_VARARGS, "setup(getDevice, getCurrentRawStream, call, require_gpu, fail)"},
    {"names", names, METH_NOARGS, "the entry points that call() knows"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_launch", "Native side of _lib.py's launch path.", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__launch() {
    s_is_cuda = PyUnicode_InternFromString("is_cuda");
    s_get_device = PyUnicode_InternFromString("get_device");
    s_data_ptr = PyUnicode_InternFromString("data_ptr");
    table = PyDict_New();
    if (!s_is_cuda || !s_get_device || !s_data_ptr || !table) return nullptr;
    for (int i = 0; i < ENTRIES; ++i) {
        PyObject* at = PyLong_FromLong(i);
        if (!at || PyDict_SetItemString(table, entries[i].name, at)) return nullptr;
        Py_DECREF(at);
    }
    return PyModule_Create(&module);
}
