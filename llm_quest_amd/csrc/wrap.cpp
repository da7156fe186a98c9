// The tensor-level launchers of kernels.py, kernels_q35.py, kernels_seq.py and ops_decode.py that a step of few rows calls by the hundred, in native code: the same checks, the same outputs, the same
// arguments to the same entry points.  A launch costs the host 3 us; in Python its checks, strides, pointers and torch.empty cost another 10 to 15, and steps of a few microseconds a kernel waited for
// them (one token of eight served sequences through four layers: 37 launches, 0.58 ms of host time over 0.38 ms of kernels).
//
// An operator here takes a call only where everything is as its Python form wants it: plain tensors of the right types, shapes and strides on the current device, no tracing or function mode.  Whatever
// else comes -- what the Python form refuses, another device, a tensor subclass, a library that is not loaded -- goes to the Python form, which stands unchanged beside it and says why.
// One CPython extension per interpreter and torch, optional: without it every call goes to Python, with the same results.
#include <torch/csrc/python_headers.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/Device.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/version.h>

#include <algorithm>
#include <initializer_list>
#include <type_traits>

#include "../../include/mi355_vlm.h"

#define WRAP_ENTRIES(E) \
    E(gemm_bf16) E(gemm_bf16_grouped_ws) E(colsum) E(rmsnorm_fwd) E(rmsnorm_bwd) E(reduce_rows_f32) E(qknorm_rope_fwd) E(qknorm_rope_bwd) E(swiglu_fwd) E(swiglu_bwd) E(attn_fwd) E(attn_bwd_ws) \
    E(attn_bwd_qnorm) E(add_f32_to_bf16) E(layernorm_fwd) E(layernorm_bwd_bf16) E(reduce_rows_into) E(reduce_rows_each) E(gelu_fwd) E(gelu_bwd_colsum) E(copy2d) E(zc_weight) E(headnorm_rope_fwd) E(headnorm_rope_bwd) \
    E(sigmoid_gate_fwd) E(sigmoid_gate_bwd) E(attn_generic_fwd) E(attn_generic_bwd) E(gdn_gates_fwd) E(gdn_gates_bwd) E(causal_conv_silu_fwd) E(causal_conv_silu_bwd) E(l2norm_fwd) E(l2norm_bwd) \
    E(gated_rmsnorm_fwd) E(gated_rmsnorm_bwd) E(gemv_bf16) E(gemv_bf16_f32out) E(hyper_mix) E(bgemm) E(latent_attn) E(qkv_rows_append) E(group_rmsnorm_sum) E(ragged_conv) E(gated_headnorm) E(glu_rows) \
    E(add_layernorm_fwd) E(rmsnorm_rows) E(latent_kv_append) E(rope_heads) E(gla_fwd) E(router_logits) E(moe_route) E(moe_dispatch) E(moe_choose) E(unary_rows) E(embed_hash_fwd)

namespace {

constexpr at::ScalarType BF16 = at::kBFloat16, F32 = at::kFloat, I32 = at::kInt, U8 = at::kByte, I64 = at::kLong;

struct Decline {};  // thrown: the call is the Python form's
struct Raised {};   // thrown: a Python exception is set

PyObject *fn_device, *fn_stream, *fn_set_device, *fn_fail;  // current device, raw handle of its stream, what launches that follow run on, raises (name, rc)
PyObject* kernels;                                          // kernels.py's namespace: its scratch and its switches
thread_local PyObject* dry;                                 // a list: this thread's calls are written there instead of made, and tensors may be anywhere (tests)

struct Slot {
    const char* name;
    void* address;
};
namespace slot {
#define E(n) Slot n{"mi355_" #n, nullptr};
WRAP_ENTRIES(E)
#undef E
}  // namespace slot
Slot* const slots[] = {
#define E(n) &slot::n,
    WRAP_ENTRIES(E)
#undef E
};
using WorkspaceBytes = int64_t (*)(int, int, int, int);
using Partials = int64_t (*)(int, int, int);
WorkspaceBytes attn_bwd_workspace_bytes;
using ChooseTakes = int (*)(int64_t, int, int, int);
ChooseTakes moe_choose_takes;
using SplitBytes = int64_t (*)(int, int, int, int, int, int);
SplitBytes attn_bwd_split_bytes;
Partials attn_bwd_qnorm_partials;

void need(bool holds) {
    if (!holds) throw Decline();
}

// a tensor argument or result; may be none
struct T {
    at::Tensor t;
    explicit operator bool() const { return t.defined(); }
    int64_t dim() const { return t.dim(); }
    int64_t size(int64_t d) const { return t.sizes()[d]; }
    int64_t ld() const { return t.defined() ? t.strides()[0] : 0; }
    int64_t numel() const { return t.numel(); }
    at::ScalarType dtype() const { return t.scalar_type(); }
    bool is(at::ScalarType s) const { return t.scalar_type() == s; }
    bool contiguous() const { return t.is_contiguous(); }
    bool rows() const { return t.dim() == 2 && t.strides()[1] == 1; }
    bool shape(std::initializer_list<int64_t> s) const { return t.sizes().equals(at::IntArrayRef(s)); }
    bool like(const T& o) const { return t.sizes().equals(o.t.sizes()); }
    bool vec(at::ScalarType s, int64_t n) const { return is(s) && contiguous() && numel() == n; }
    bool vec_or_none(at::ScalarType s, int64_t n) const { return !t.defined() || vec(s, n); }
    int code() const {  // 0 for none, as the launchers pass it
        if (!t.defined()) return MI355_DT_BF16;
        need(is(BF16) || is(F32));
        return is(BF16) ? MI355_DT_BF16 : MI355_DT_F32;
    }
    void* ptr() const { return t.defined() ? t.data_ptr() : nullptr; }
    uintptr_t addr() const { return reinterpret_cast<uintptr_t>(ptr()); }
};
int code(at::ScalarType s) {
    need(s == BF16 || s == F32);
    return s == BF16 ? MI355_DT_BF16 : MI355_DT_F32;
}

PyObject* wrapped(const T& t) {
    if (!t.t.defined()) Py_RETURN_NONE;
    return THPVariable_Wrap(t.t);
}
template <class... A>
PyObject* tuple(const A&... a) {  // steals nothing; tensors, none
    PyObject* out = PyTuple_New(sizeof...(a));
    if (!out) throw Raised();
    Py_ssize_t i = 0;
    PyObject* items[] = {wrapped(a)...};
    for (PyObject* o : items) PyTuple_SET_ITEM(out, i++, o);
    return out;
}

PyObject* item(PyObject* space, const char* name) {  // borrowed
    PyObject* o = space ? PyDict_GetItemString(space, name) : nullptr;
    need(o != nullptr);
    return o;
}
long number(PyObject* o) {
    const long v = PyLong_AsLong(o);
    if (v == -1 && PyErr_Occurred()) PyErr_Clear(), throw Decline();
    return v;
}
PyObject* kernels_item(const char* name) { return item(kernels, name); }
long kernels_int(const char* name) { return number(kernels_item(name)); }
bool kernels_true(const char* name) { return PyObject_IsTrue(kernels_item(name)) == 1; }

constexpr int MAX_ARGS = 34;

struct Call {
    PyObject* v[MAX_ARGS] = {};
    PyObject* home = nullptr;  // the namespace of the Python form, whose constants hold here too
    int device = -1;
    bool ready = false;
    void* stream = nullptr;

    long constant(const char* name) const { return number(item(home, name)); }
    bool given(int i) const { return v[i] && v[i] != Py_None; }
    T tensor(int i) {
        T t = maybe(i);
        need(t.t.defined());
        return t;
    }
    T maybe(int i) { return from(v[i]); }
    T from(PyObject* o) {
        if (!o || o == Py_None) return T{};
        need(THPVariable_CheckExact(o));  // (a subclass may mean anything by its methods)
        const at::Tensor& t = THPVariable_Unpack(o);
        need(t.defined() && t.layout() == at::kStrided && t.has_storage() && !t.key_set().has(c10::DispatchKey::Python));
        if (!dry) {
            need(t.is_cuda());
            const int d = t.get_device();
            need(device < 0 || d == device);
            device = d;
        }
        return T{t};
    }
    int64_t integer(int i, int64_t otherwise) const { return v[i] ? integer(i) : otherwise; }
    int64_t integer(int i) const {
        need(v[i] && PyLong_Check(v[i]));
        int over = 0;
        const int64_t x = PyLong_AsLongLongAndOverflow(v[i], &over);
        need(!over);
        return x;
    }
    double real(int i, double otherwise) const { return v[i] ? real(i) : otherwise; }
    double real(int i) const {
        need(v[i] != nullptr);
        if (PyFloat_CheckExact(v[i])) return PyFloat_AS_DOUBLE(v[i]);
        return static_cast<double>(integer(i));
    }
    bool truth(int i, bool otherwise) const {
        if (!v[i]) return otherwise;
        need(PyBool_Check(v[i]) || PyLong_CheckExact(v[i]));
        return PyObject_IsTrue(v[i]) == 1;
    }
    at::ScalarType dtype(int i, at::ScalarType otherwise) const {
        if (!given(i)) return otherwise;
        need(THPDtype_Check(v[i]));
        return reinterpret_cast<THPDtype*>(v[i])->scalar_type;
    }

    T empty(const T& beside, at::IntArrayRef sizes, at::ScalarType s) {
        need(s == BF16 || s == F32 || s == I32);
        return T{at::empty(sizes, beside.t.options().dtype(s).requires_grad(false))};
    }
    T empty_like(const T& t) { return T{at::empty_like(t.t)}; }

    void get_ready() {  // where the launches go: the operands' device, if it is the current one
        if (ready) return;
        need(device >= 0);
        PyObject* cur = PyObject_CallNoArgs(fn_device);
        if (!cur) throw Raised();
        const long at = PyLong_AsLong(cur);
        if (at != device) Py_DECREF(cur), throw Decline();
        PyObject* set = fn_set_device ? PyObject_CallOneArg(fn_set_device, cur) : Py_NewRef(Py_None);  // as after require_gpu of these operands
        PyObject* h = set ? PyObject_CallOneArg(fn_stream, cur) : nullptr;
        Py_XDECREF(set);
        Py_DECREF(cur);
        if (!h) throw Raised();
        stream = PyLong_AsVoidPtr(h);
        Py_DECREF(h);
        if (PyErr_Occurred()) throw Raised();
        ready = true;
    }

    template <class P>
    static P as(const T& t) { return reinterpret_cast<P>(t.ptr()); }
    template <class P, class A, std::enable_if_t<!std::is_same_v<A, T>, int> = 0>
    static P as(A a) {
        if constexpr (std::is_pointer_v<P> && std::is_integral_v<A>) return reinterpret_cast<P>(static_cast<uintptr_t>(a));
        else return static_cast<P>(a);
    }
    template <class P>
    static PyObject* shown(P p) {
        if constexpr (std::is_pointer_v<P>) return p ? PyLong_FromUnsignedLongLong(reinterpret_cast<uintptr_t>(p)) : Py_NewRef(Py_None);
        else if constexpr (std::is_floating_point_v<P>) return PyFloat_FromDouble(p);
        else return PyLong_FromLongLong(p);
    }
    template <class... P, class... A>
    void launch(const Slot& s, int (*)(P...), const A&... args) {
        if (dry) return record(s, static_cast<void (*)(P...)>(nullptr), args...);
        need(s.address != nullptr);
        get_ready();
        int rc;
        invoke(s, rc, static_cast<int (*)(P...)>(nullptr), args...);
        if (rc != 0) fail(s, rc);
    }
    template <class... P, class... A>
    void invoke(const Slot& s, int& rc, int (*)(P...), const A&... args) {
        call_as<P...>(s, rc, args..., stream);
    }
    template <class... P, class... A>
    void call_as(const Slot& s, int& rc, const A&... args) {
        static_assert(sizeof...(P) == sizeof...(A), "an entry point's arguments, without the stream");
        std::tuple<P...> all{as<P>(args)...};  // (every pointer is read with the interpreter's lock held)
        Py_BEGIN_ALLOW_THREADS
        rc = std::apply(reinterpret_cast<int (*)(P...)>(s.address), all);
        Py_END_ALLOW_THREADS
    }
    template <class... P, class... A>
    void record(const Slot& s, void (*)(P...), const A&... args) {
        show_as<P...>(s, args..., static_cast<void*>(nullptr));
    }
    template <class... P, class... A>
    void show_as(const Slot& s, const A&... args) {
        static_assert(sizeof...(P) == sizeof...(A), "an entry point's arguments, without the stream");
        PyObject* items[] = {PyUnicode_FromString(s.name), shown<P>(as<P>(args))...};
        PyObject* row = PyTuple_New(sizeof...(P));  // the name, the arguments without the stream
        for (size_t i = 0; i < sizeof...(P); ++i) PyTuple_SET_ITEM(row, i, items[i]);
        Py_DECREF(items[sizeof...(P)]);
        PyList_Append(dry, row);
        Py_DECREF(row);
    }
    [[noreturn]] void fail(const Slot& s, int rc) {
        PyObject* r = PyObject_CallFunction(fn_fail, "si", s.name, rc);
        Py_XDECREF(r);
        if (!PyErr_Occurred()) PyErr_Format(PyExc_RuntimeError, "%s failed (rc=%d)", s.name, rc);
        throw Raised();
    }

    // scratch of the (device, stream), kept by kernels.py
    T workspace(const T& beside) {
        PyObject* dev = THPDevice_New(beside.t.device());
        if (!dev) throw Raised();
        PyObject* got = nullptr;
        if (!dry) {
            get_ready();
            PyObject* h = PyLong_FromVoidPtr(stream);
            PyObject* key = h ? PyTuple_Pack(2, dev, h) : nullptr;
            Py_XDECREF(h);
            if (!key) Py_DECREF(dev), throw Raised();
            PyObject* all = kernels_item("_WS");
            got = PyDict_GetItemWithError(all, key);
            Py_XINCREF(got);
            Py_DECREF(key);
            if (!got && PyErr_Occurred()) Py_DECREF(dev), throw Raised();
        }
        if (!got) got = PyObject_CallOneArg(kernels_item("_workspace"), dev);
        Py_DECREF(dev);
        if (!got) throw Raised();
        T t{THPVariable_Unpack(got)};
        Py_DECREF(got);
        return t;
    }
};
#define LAUNCH(entry, ...) c.launch(slot::entry, static_cast<decltype(&mi355_##entry)>(nullptr), __VA_ARGS__)

struct Op {
    const char* name;
    const char* const* args;
    int n;
    PyObject* (*body)(Call&);
    PyObject* interned[MAX_ARGS];
};
Op ops[64];
int n_ops = 0;
struct Registered {
    Registered(const char* name, const char* const* args, int n, PyObject* (*body)(Call&)) { ops[n_ops++] = Op{name, args, n, body, {}}; }
};
#define OP(op, ...)                                                                                            \
    const char* const op##_args[] = {__VA_ARGS__};                                                             \
    static_assert(sizeof(op##_args) / sizeof(char*) <= MAX_ARGS, "raise MAX_ARGS");                            \
    PyObject* op##_body(Call& c);                                                                              \
    const Registered op##_registered(#op, op##_args, static_cast<int>(sizeof(op##_args) / sizeof(char*)), op##_body); \
    PyObject* op##_body(Call& c)

// ---------------------------------------------------------------------------------------------- kernels.py
// product with the checks of kernels.gemm; no tile hint, no split3 output.  A launch that a window of kernels.py counts goes to Python (see _nt_tick).
T product(Call& c, int form, const T& a, const T& b, T out, at::ScalarType out_dtype, const T& bias, const T& residual, int epilogue, bool may_split) {
    need(a.rows() && b.rows() && a.is(BF16) && b.is(BF16));
    const bool at = form == MI355_GEMM_TN, bt = form != MI355_GEMM_NT;
    const int64_t M = a.size(at), K = a.size(!at), N = b.size(bt), K2 = b.size(!bt);
    need(K == K2);
    if (!out) out = c.empty(a, {M, N}, out_dtype);
    need(out.rows() && out.shape({M, N}));
    need(!bias || (bias.is(F32) && bias.numel() == N && bias.contiguous()));
    need(!residual || (residual.rows() && residual.dtype() == out.dtype() && residual.shape({M, N})));
    need(kernels_int("_TILE_OVERRIDE") == 0 && kernels_int("_TILE_NT_PLAIN") == 0);
    PyObject* key = PyLong_FromLong(form);
    PyObject* tile = PyDict_GetItem(kernels_item("_TILE_BY_FORM"), key);
    Py_DECREF(key);
    need(tile && PyLong_Check(tile) && PyLong_AsLong(tile) == 0);
    if (form == MI355_GEMM_NT && out.is(BF16) && !bias && epilogue == MI355_EPI_NONE && K % 64 == 0 && K >= 128)
        need(kernels_item("_PERSIST_USER") == Py_None && ((M + 255) / 256) * ((N + 255) / 256) < kernels_int("PERSIST_MIN_TILES"));
    T ws;
    if (may_split) ws = c.workspace(a);
    LAUNCH(gemm_bf16, form, M, N, K, a, a.ld(), b, b.ld(), out, out.ld(), out.code(), bias, residual, residual.ld(), epilogue, ws, may_split ? kernels_int("WS_BYTES") : 0L, 0);
    return out;
}

OP(gemm, "form", "a", "b", "out", "out_dtype", "bias", "residual", "gelu", "allow_split_k", "tile", "split3_out") {
    need(!c.truth(10, false) && c.integer(9, 0) == 0);
    const T a = c.tensor(1), b = c.tensor(2), out = c.maybe(3), bias = c.maybe(5), residual = c.maybe(6);
    const int64_t form = c.integer(0);
    need(form >= 0 && form <= 2 && (!c.v[4] || c.given(4)));
    return wrapped(product(c, (int)form, a, b, out, c.dtype(4, BF16), bias, residual, c.truth(7, false) ? MI355_EPI_GELU_ERF : MI355_EPI_NONE, c.truth(8, true)));
}

OP(dgrad, "dy", "w", "out") {
    const T dy = c.tensor(0), w = c.tensor(1), out = c.maybe(2);
    need(dy.rows() && dy.size(0) < std::min(c.constant("DGRAD_NT_MIN_ROWS"), 1280L));  // (kernels.dgrad_transposes says no to fewer rows than both)
    return wrapped(product(c, MI355_GEMM_NN, dy, w, out, BF16, T{}, T{}, MI355_EPI_NONE, true));
}

OP(gemm_gateup_swiglu, "x", "w_fused", "tile") {
    const T x = c.tensor(0), w = c.tensor(1);
    need(c.integer(2, 0) == 0 && x.rows() && w.rows());
    const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
    need(x.is(BF16) && w.is(BF16) && w.size(1) == K && N % 64 == 0 && kernels_int("_TILE_OVERRIDE") == 0 && kernels_int("_TILE_SWIGLU_FWD") == 0);
    need(kernels_item("_PERSIST_USER") == Py_None && ((M + 255) / 256) * ((N + 255) / 256) < kernels_int("PERSIST_MIN_TILES"));
    PyObject* key = PyLong_FromLong(MI355_GEMM_NT);
    PyObject* tile = PyDict_GetItem(kernels_item("_TILE_BY_FORM"), key);
    Py_DECREF(key);
    need(tile && PyLong_Check(tile) && PyLong_AsLong(tile) == 0);
    const T gu = c.empty(x, {M, N}, BF16), a = c.empty(x, {M, N / 2}, BF16);
    LAUNCH(gemm_bf16, MI355_GEMM_NT, M, N, K, x, x.ld(), w, w.ld(), gu, gu.ld(), MI355_DT_BF16, T{}, a, a.ld(), MI355_EPI_SWIGLU_FWD, T{}, 0, 0);
    return tuple(gu, a);
}

OP(gemm_dgrad_swiglu_bwd, "dy", "w", "gu", "tile") {
    const T dy = c.tensor(0), w = c.tensor(1), gu = c.tensor(2);
    need(c.integer(3, 0) == 0 && dy.rows() && w.rows());
    const int64_t M = dy.size(0), K = dy.size(1), F = w.size(1);
    need(dy.is(BF16) && w.is(BF16) && gu.is(BF16) && w.size(0) == K && gu.contiguous() && gu.shape({M, 2 * F}) && kernels_int("_TILE_OVERRIDE") == 0);
    need(M < kernels_int("DGRAD_NT_MIN_ROWS") && kernels_true("DGRAD_NT"));  // (from there on kernels.dgrad_on_quad decides about the form)
    PyObject* key = PyLong_FromLong(MI355_GEMM_NN);
    PyObject* tile = PyDict_GetItem(kernels_item("_TILE_BY_FORM"), key);
    Py_DECREF(key);
    need(tile && PyLong_Check(tile) && PyLong_AsLong(tile) == 0);
    const T out = c.empty_like(gu);
    LAUNCH(gemm_bf16, MI355_GEMM_NN, M, F, K, dy, dy.ld(), w, w.ld(), out, out.ld(), MI355_DT_BF16, T{}, gu, gu.ld(), MI355_EPI_SWIGLU_BWD, T{}, 0, 0);
    return wrapped(out);
}

OP(colsum, "x", "out", "accumulate") {
    const T x = c.tensor(0);
    T out = c.maybe(1);
    need(x.rows());
    if (!out) out = c.empty(x, {x.size(1)}, F32);
    need(out.is(F32) && out.numel() == x.size(1) && out.contiguous());
    LAUNCH(colsum, x.size(0), x.size(1), x, x.code(), x.ld(), out, (int)c.truth(2, false));
    return wrapped(out);
}

OP(rmsnorm_fwd, "x2d", "w", "eps", "want_rstd") {
    const T x = c.tensor(0), w = c.tensor(1);
    need(x.dim() == 2 && x.is(BF16) && w.is(BF16) && x.contiguous() && w.numel() == x.size(1));
    const T y = c.empty_like(x), rstd = c.truth(3, true) ? c.empty(x, {x.size(0)}, F32) : T{};
    LAUNCH(rmsnorm_fwd, x.size(0), x.size(1), x, w, y, rstd, c.real(2, 1e-6));
    return tuple(y, rstd);
}

OP(rmsnorm_bwd, "x2d", "w", "rstd", "dy", "dres", "dw_out", "dw_accumulate", "partial") {
    const T x = c.tensor(0), w = c.tensor(1), rstd = c.tensor(2), dy = c.tensor(3), dres = c.maybe(4);
    T dw = c.maybe(5);
    need(x.dim() == 2 && dy.contiguous() && dy.like(x) && dy.is(BF16) && (!dres || (dres.contiguous() && dres.like(x) && dres.is(BF16))));
    const int64_t rows = x.size(0), width = x.size(1), parts = std::min<int64_t>(c.constant("NORM_PARTS"), (rows + 3) / 4);
    const bool accumulate = c.truth(6, false) && dw;
    const int dw_code = dw ? dw.code() : MI355_DT_F32;
    const T dx = c.empty_like(x), part = c.empty(x, {parts, width}, F32);
    need(dry || slot::reduce_rows_f32.address);
    LAUNCH(rmsnorm_bwd, rows, width, x, w, rstd, dy, dres, dx, part, parts);
    if (c.truth(7, false)) return tuple(dx, part);
    if (!dw) dw = c.empty(x, {width}, F32);
    LAUNCH(reduce_rows_f32, parts, width, part, dw, dw_code, (int)accumulate);
    return tuple(dx, dw);
}

OP(qknorm_rope_fwd, "qkv", "qw", "kw", "cos", "sin", "pos", "Hq", "Hkv", "D", "eps") {
    const T qkv = c.tensor(0), qw = c.maybe(1), kw = c.maybe(2), cos = c.tensor(3), sin = c.tensor(4), pos = c.tensor(5);
    const int64_t Hq = c.integer(6), Hkv = c.integer(7), D = c.integer(8);
    need(qkv.dim() == 2 && qkv.contiguous() && qkv.is(BF16) && qkv.size(1) == (Hq + 2 * Hkv) * D && cos.is(F32) && sin.is(F32) && cos.contiguous() && sin.contiguous() && cos.dim() == 2 && cos.size(1) == D);
    const int64_t tokens = qkv.size(0);
    need(pos.vec(I32, tokens));
    const T q = c.empty(qkv, {tokens, Hq * D}, BF16), k = c.empty(qkv, {tokens, Hkv * D}, BF16), rstd = qw ? c.empty(qkv, {tokens, Hq + Hkv}, F32) : T{};
    LAUNCH(qknorm_rope_fwd, tokens, Hq, Hkv, D, qkv, qw, kw, cos, sin, pos, q, k, rstd, c.real(9, 1e-6));
    return tuple(q, k, rstd);
}

OP(qknorm_rope_bwd, "qkv", "qw", "kw", "cos", "sin", "pos", "rstd", "dq", "dk", "dqkv", "Hq", "Hkv", "D", "partial") {
    const T qkv = c.tensor(0), qw = c.maybe(1), kw = c.maybe(2), cos = c.maybe(3), sin = c.maybe(4), pos = c.maybe(5), rstd = c.maybe(6), dq = c.maybe(7), dk = c.tensor(8), dqkv = c.tensor(9);
    const int64_t Hq = c.integer(10), Hkv = c.integer(11), D = c.integer(12);
    need(qkv.dim() == 2);
    const int64_t tokens = qkv.size(0), hpw = D == 128 ? 4 : 8;
    need(!dq || (dq.contiguous() && dq.is(BF16) && dq.shape({tokens, Hq * D})));
    need(dk.contiguous() && dk.is(BF16) && dk.shape({tokens, Hkv * D}) && dqkv.contiguous() && dqkv.like(qkv) && dqkv.is(BF16));
    const int64_t parts = std::min<int64_t>(c.constant("QK_PARTS"), (tokens * ((Hq + Hkv + hpw - 1) / hpw) + 3) / 4);
    const T part = c.empty(qkv, {parts, 2 * D}, F32);
    need(dry || slot::reduce_rows_f32.address);
    LAUNCH(qknorm_rope_bwd, tokens, Hq, Hkv, D, qkv, qw, kw, cos, sin, pos, rstd, dq, dk, dqkv, part, parts);
    if (c.truth(13, false)) return tuple(T{part.t.narrow(1, 0, D)}, T{part.t.narrow(1, D, D)});
    const T dw = c.empty(qkv, {2 * D}, F32);
    LAUNCH(reduce_rows_f32, parts, 2 * D, part, dw, MI355_DT_F32, 0);
    return tuple(T{dw.t.narrow(0, 0, D)}, T{dw.t.narrow(0, D, D)});
}

OP(swiglu_fwd, "gu", "F") {
    const T gu = c.tensor(0);
    const int64_t F = c.integer(1);
    need(gu.dim() == 2 && gu.contiguous() && gu.is(BF16) && gu.size(1) == 2 * F);
    const T a = c.empty(gu, {gu.size(0), F}, BF16);
    LAUNCH(swiglu_fwd, gu.size(0), F, gu, a);
    return wrapped(a);
}

OP(swiglu_bwd, "gu", "da", "F") {
    const T gu = c.tensor(0), da = c.tensor(1);
    const int64_t F = c.integer(2);
    need(gu.dim() >= 1 && da.contiguous() && da.is(BF16) && da.shape({gu.size(0), F}));
    const T dgu = c.empty_like(gu);
    LAUNCH(swiglu_bwd, gu.size(0), F, gu, da, dgu);
    return wrapped(dgu);
}

bool attn_operand(const T& t, int64_t tokens, int64_t width) { return t.is(BF16) && t.rows() && t.size(0) == tokens && t.size(1) == width; }

OP(attn_fwd, "q", "k", "v", "B", "S", "Hq", "Hkv", "D", "key_mask", "causal", "scale") {
    const T q = c.tensor(0), k = c.tensor(1), v = c.tensor(2), mask = c.maybe(8);
    const int64_t B = c.integer(3), S = c.integer(4), Hq = c.integer(5), Hkv = c.integer(6), D = c.integer(7);
    need(D > 0 && attn_operand(q, B * S, Hq * D) && attn_operand(k, B * S, Hkv * D) && attn_operand(v, B * S, Hkv * D) && (!mask || (mask.is(U8) && mask.contiguous() && mask.shape({B, S}))));
    const double scale = c.given(10) ? c.real(10) : std::pow((double)D, -0.5);
    const T o = c.empty(q, {B * S, Hq * D}, BF16), lse = c.empty(q, {B, Hq, S}, F32);
    LAUNCH(attn_fwd, B, S, Hq, Hkv, D, q, q.ld(), k, k.ld(), v, v.ld(), o, o.ld(), lse, mask, (int)c.truth(9, true) | kernels_int("_ATTN_ABLATE"), scale);
    return tuple(o, lse);
}

// kernels._attn_scratch(device, bytes): a tensor, or none where it gives none
T attn_scratch(Call& c, const T& beside, int64_t bytes) {
    PyObject* dev = THPDevice_New(beside.t.device());
    if (!dev) throw Raised();
    PyObject* n = PyLong_FromLongLong(bytes);
    PyObject* got = n ? PyObject_CallFunctionObjArgs(kernels_item("_attn_scratch"), dev, n, nullptr) : nullptr;
    Py_DECREF(dev);
    Py_XDECREF(n);
    if (!got) throw Raised();
    T t = got == Py_None ? T{} : T{THPVariable_Unpack(got)};
    Py_DECREF(got);
    return t;
}
// kernels._attn_split_scratch: `bytes` and room for the parts of split key blocks, or `bytes` alone
T attn_split_scratch(Call& c, const T& beside, int64_t& bytes, int B, int S, int Hq, int Hkv, int D, int causal) {
    if (const int64_t more = attn_bwd_split_bytes(B, S, Hq, Hkv, D, causal))
        if (T t = attn_scratch(c, beside, bytes + more)) {
            bytes += more;
            return t;
        }
    return attn_scratch(c, beside, bytes);
}
void count_form(const char* form) {  // kernels.attn_bwd_form[form] += 1
    PyObject* all = kernels_item("attn_bwd_form");
    PyObject* n = PyDict_GetItemString(all, form);
    PyObject* m = PyLong_FromLong(n ? PyLong_AsLong(n) + 1 : 1);
    if (m) PyDict_SetItemString(all, form, m), Py_DECREF(m);
}

OP(attn_bwd, "q", "k", "v", "o", "do", "lse", "B", "S", "Hq", "Hkv", "D", "dq", "dk", "dv", "key_mask", "causal", "scale") {
    const T q = c.tensor(0), k = c.tensor(1), v = c.tensor(2), o = c.tensor(3), dO = c.tensor(4), lse = c.tensor(5), dq = c.tensor(11), dk = c.tensor(12), dv = c.tensor(13), mask = c.maybe(14);
    const int64_t B = c.integer(6), S = c.integer(7), Hq = c.integer(8), Hkv = c.integer(9), D = c.integer(10);
    need(D > 0);
    for (const T* t : {&q, &o, &dO, &dq}) need(attn_operand(*t, B * S, Hq * D));
    for (const T* t : {&k, &v, &dk, &dv}) need(attn_operand(*t, B * S, Hkv * D));
    need(lse.is(F32) && lse.contiguous() && lse.shape({B, Hq, S}) && attn_bwd_workspace_bytes && attn_bwd_split_bytes && (dry || slot::attn_bwd_ws.address));
    const double scale = c.given(16) ? c.real(16) : std::pow((double)D, -0.5);
    const int flags = (int)c.truth(15, true) | (int)kernels_int("_ATTN_ABLATE");
    const T delta = c.empty_like(lse);
    int64_t bytes = kernels_true("_ATTN_DS_SPILL") ? attn_bwd_workspace_bytes(B, S, Hq, D) : 0;
    T ws;
    if (!dry) c.get_ready();
    if (bytes) {
        ws = attn_split_scratch(c, q, bytes, B, S, Hq, Hkv, D, c.truth(15, true));
        if (!ws) bytes = 0;  // (over the cap, or no memory: the recompute form)
    }
    count_form(bytes ? "spill" : "recompute");
    LAUNCH(attn_bwd_ws, B, S, Hq, Hkv, D, q, q.ld(), k, k.ld(), v, v.ld(), o, o.ld(), dO, dO.ld(), lse, delta, dq, dq.ld(), dk, dk.ld(), dv, dv.ld(), mask, flags, scale, ws, bytes);
    Py_RETURN_NONE;
}

OP(attn_bwd_qnorm, "q", "k", "v", "o", "do", "lse", "B", "S", "Hq", "Hkv", "D", "dk", "dv", "qkv", "qw", "cos", "sin", "pos", "rstd", "dqkv", "key_mask", "causal", "scale", "delta", "partial") {
    const int64_t B = c.integer(6), S = c.integer(7), Hq = c.integer(8), Hkv = c.integer(9), D = c.integer(10);
    need(D == 128 && c.given(14) && kernels_true("FUSE_QNORM_BWD") && kernels_true("_ATTN_DS_SPILL"));
    const T q = c.tensor(0), k = c.tensor(1), v = c.tensor(2), o = c.tensor(3), dO = c.tensor(4), lse = c.tensor(5), dk = c.tensor(11), dv = c.tensor(12), qkv = c.tensor(13), qw = c.tensor(14), cos = c.tensor(15),
            sin = c.tensor(16), pos = c.tensor(17), rstd = c.tensor(18), dqkv = c.tensor(19), mask = c.maybe(20);
    T delta = c.maybe(23);
    for (const T* t : {&q, &o, &dO}) need(attn_operand(*t, B * S, Hq * D));
    for (const T* t : {&k, &v, &dk, &dv}) need(attn_operand(*t, B * S, Hkv * D));
    need(lse.is(F32) && lse.contiguous() && lse.shape({B, Hq, S}) && qkv.is(BF16) && dqkv.is(BF16) && qkv.like(dqkv) && qkv.rows() && dqkv.rows() && qkv.size(0) == B * S);
    need(rstd.is(F32) && rstd.dim() == 2 && rstd.contiguous() && rstd.size(0) == B * S && rstd.size(1) >= Hq && qw.is(BF16) && qw.numel() == D);
    need(cos.is(F32) && sin.is(F32) && cos.contiguous() && sin.contiguous() && cos.dim() >= 1 && cos.size(cos.dim() - 1) == D && pos.is(I32) && pos.numel() == B * S);
    need(!delta || (delta.is(F32) && delta.contiguous() && delta.like(lse)));
    need(attn_bwd_workspace_bytes && attn_bwd_split_bytes && attn_bwd_qnorm_partials && (dry || (slot::attn_bwd_qnorm.address && slot::reduce_rows_f32.address)));
    const double scale = c.given(22) ? c.real(22) : std::pow((double)D, -0.5);
    int flags = (int)c.truth(21, true) | (int)kernels_int("_ATTN_ABLATE");
    if (!dry) c.get_ready();
    int64_t bytes = attn_bwd_workspace_bytes(B, S, Hq, D);
    const T ws = !bytes ? T{} : delta ? attn_scratch(c, q, bytes) : attn_split_scratch(c, q, bytes, B, S, Hq, Hkv, D, c.truth(21, true));
    need(bool(ws));
    PyObject* cs = PyObject_CallFunctionObjArgs(kernels_item("rope_cs16"), c.v[15], c.v[16], nullptr);
    if (!cs) throw Raised();
    T cs16;
    if (cs != Py_None) cs16 = T{THPVariable_Unpack(cs)};
    Py_DECREF(cs);
    count_form("spill");
    if (delta) flags |= MI355_ATTN_DELTA_READY;
    else delta = c.empty_like(lse);
    const int64_t parts = attn_bwd_qnorm_partials(B, S, Hq);
    const T part = c.empty(q, {parts, D}, F32);
    LAUNCH(attn_bwd_qnorm, B, S, Hq, Hkv, D, q, q.ld(), k, k.ld(), v, v.ld(), o, o.ld(), dO, dO.ld(), lse, delta, dk, dk.ld(), dv, dv.ld(), mask, flags, scale, ws, bytes, qkv, qkv.ld(), qw, cos, sin, pos, rstd,
           rstd.size(1), dqkv, dqkv.ld(), part, cs16);
    const bool partial = c.truth(24, false);
    const T dw = partial ? T{} : c.empty(q, {D}, F32);  // one partial row per workgroup: summed in two fixed-order levels
    int64_t fold = 1;
    for (int64_t f : {64, 32, 16, 8})
        if (fold == 1 && parts % f == 0 && parts / f >= 8) fold = f;
    if (fold > 1) {
        const T mid = c.empty(q, {fold * D}, F32);
        LAUNCH(reduce_rows_f32, parts / fold, fold * D, part, mid, MI355_DT_F32, 0);
        if (partial) return wrapped(T{mid.t.view({fold, D})});
        LAUNCH(reduce_rows_f32, fold, D, mid, dw, MI355_DT_F32, 0);
    } else {
        if (partial) return wrapped(part);
        LAUNCH(reduce_rows_f32, parts, D, part, dw, MI355_DT_F32, 0);
    }
    return wrapped(dw);
}

OP(add_f32_to_bf16, "a_f32", "b_bf16", "dst_bf16") {
    const T a = c.tensor(0), b = c.maybe(1), d = c.tensor(2);
    LAUNCH(add_f32_to_bf16, a.numel(), a, b, d);
    Py_RETURN_NONE;
}

OP(layernorm_fwd, "x2d", "scale", "shift", "out_dtype", "eps", "want_stats", "mode") {
    const T x = c.tensor(0), scale = c.tensor(1), shift = c.tensor(2);
    const at::ScalarType od = c.dtype(3, BF16);
    const bool stats = c.truth(5, false);
    need((!c.v[3] || c.given(3)) && x.dim() == 2 && x.is(F32) && x.contiguous() && scale.is(F32) && shift.is(F32));
    const T y = c.empty(x, {x.size(0), x.size(1)}, od), mean = stats ? c.empty(x, {x.size(0)}, F32) : T{}, rsig = stats ? c.empty_like(mean) : T{};
    LAUNCH(layernorm_fwd, x.size(0), x.size(1), x, scale, shift, y, code(od), mean, rsig, c.real(4, 1e-5), c.integer(6, 0));
    return stats ? tuple(y, mean, rsig) : wrapped(y);
}

// kernels.reduce_rows_into(partial, parts, width, dests) for destinations of which none comes twice
struct Dests {
    T t[4];
    int n = 0, accumulate = 0;
};
Dests destinations(Call& c, PyObject* seq, int64_t width) {
    need(PyTuple_CheckExact(seq) || PyList_CheckExact(seq));
    Dests d;
    d.n = (int)PySequence_Fast_GET_SIZE(seq);
    need(d.n >= 1 && d.n <= 4);
    bool any = false;
    for (int i = 0; i < d.n; ++i) {
        PyObject* o = PySequence_Fast_GET_ITEM(seq, i);
        if (o == Py_None) continue;
        need(PyTuple_CheckExact(o) && PyTuple_GET_SIZE(o) == 2);
        PyObject* acc = PyTuple_GET_ITEM(o, 1);
        need(PyBool_Check(acc));
        d.t[i] = c.from(PyTuple_GET_ITEM(o, 0));
        need(bool(d.t[i]) && d.t[i].vec(F32, width));
        for (int j = 0; j < i; ++j) need(!d.t[j] || d.t[j].ptr() != d.t[i].ptr());
        if (acc == Py_True) d.accumulate |= 1 << i;
        any = true;
    }
    need(any);
    return d;
}

OP(reduce_rows_each, "sums") {
    need(c.v[0] && PyList_CheckExact(c.v[0]));
    const int n = (int)PyList_GET_SIZE(c.v[0]);
    need(n >= 1 && n <= 4);
    T part[4], out[4];
    int64_t parts[4] = {}, width[4] = {}, ld[4] = {}, flags[4] = {};
    for (int i = 0; i < n; ++i) {
        PyObject* q = PyList_GET_ITEM(c.v[0], i);
        need(PyTuple_CheckExact(q) && PyTuple_GET_SIZE(q) == 3 && PyBool_Check(PyTuple_GET_ITEM(q, 2)));
        part[i] = c.from(PyTuple_GET_ITEM(q, 0)), out[i] = c.from(PyTuple_GET_ITEM(q, 1));
        need(part[i] && out[i] && part[i].rows() && part[i].is(F32) && part[i].numel() > 0 && out[i].contiguous() && out[i].numel() == part[i].size(1));
        parts[i] = part[i].size(0), width[i] = part[i].size(1), ld[i] = parts[i] > 1 ? part[i].ld() : width[i];
        flags[i] = (code(out[i].dtype()) == MI355_DT_BF16 ? 1 : 0) | (PyTuple_GET_ITEM(q, 2) == Py_True ? 2 : 0);
    }
    LAUNCH(reduce_rows_each, part[0], ld[0], parts[0], width[0], out[0], flags[0], part[1], ld[1], parts[1], width[1], out[1], flags[1], part[2], ld[2], parts[2], width[2], out[2], flags[2], part[3],
           ld[3], parts[3], width[3], out[3], flags[3]);
    Py_RETURN_NONE;
}

OP(reduce_rows_into, "partial", "parts", "width", "dests") {
    const T partial = c.tensor(0);
    const int64_t width = c.integer(2);
    need(c.v[3]);
    const Dests d = destinations(c, c.v[3], width);
    LAUNCH(reduce_rows_into, c.integer(1), d.n, width, partial, d.t[0], d.t[1], d.t[2], d.t[3], d.accumulate);
    Py_RETURN_NONE;
}

OP(layernorm_bwd_bf16, "x2d", "scale", "mean", "rsig", "dy", "dres", "dests", "eps", "mode") {
    const T x = c.tensor(0), scale = c.tensor(1), mean = c.tensor(2), rsig = c.tensor(3), dy = c.tensor(4), dres = c.maybe(5);
    need(x.dim() == 2 && x.is(F32) && x.contiguous() && dy.contiguous() && dy.like(x) && (!dres || (dres.is(F32) && dres.contiguous() && dres.like(x))) && c.v[6]);
    const int64_t rows = x.size(0), width = x.size(1), parts = std::min<int64_t>(1024, (rows + 3) / 4);
    const int dyc = dy.code();
    const Dests d = destinations(c, c.v[6], width);
    need(d.n == 3 && (dry || slot::reduce_rows_into.address));
    const double eps = c.real(7, 1e-5);
    const int64_t mode = c.integer(8, 0);
    const T dx = c.empty_like(x), dxb = c.empty(x, {rows, width}, BF16), part = c.empty(x, {parts, 3 * width}, F32);
    LAUNCH(layernorm_bwd_bf16, rows, width, x, scale, mean, rsig, dy, dyc, dres, dx, dxb, part, parts, eps, mode);
    LAUNCH(reduce_rows_into, parts, d.n, width, part, d.t[0], d.t[1], d.t[2], d.t[3], d.accumulate);
    return tuple(dx, dxb);
}

OP(gelu_fwd, "x", "tanh") {
    const T x = c.tensor(0);
    need(x.is(BF16) && x.contiguous() && x.numel() % 8 == 0);
    const T y = c.empty_like(x);
    LAUNCH(gelu_fwd, x.numel(), x, y, (int)c.truth(1, false));
    return wrapped(y);
}

OP(gelu_bwd_colsum, "x", "dy", "dest", "tanh") {
    const T x = c.tensor(0), dy = c.tensor(1);
    need(x.is(BF16) && dy.is(BF16) && x.dim() == 2 && x.contiguous() && dy.contiguous() && dy.like(x) && x.size(1) % 8 == 0 && c.v[2]);
    const int64_t rows = x.size(0), width = x.size(1), parts = std::max<int64_t>(1, std::min<int64_t>(256, rows / 32));
    PyObject* one = PyTuple_Pack(1, c.v[2]);
    if (!one) throw Raised();
    Dests d;
    try {
        d = destinations(c, one, width);
    } catch (...) {
        Py_DECREF(one);
        throw;
    }
    Py_DECREF(one);
    need(dry || slot::reduce_rows_into.address);
    const int tanh = c.truth(3, false);
    const T dx = c.empty_like(x), part = c.empty(x, {parts, width}, F32);
    LAUNCH(gelu_bwd_colsum, rows, width, x, dy, dx, part, parts, tanh);
    LAUNCH(reduce_rows_into, parts, 1, width, part, d.t[0], T{}, T{}, T{}, d.accumulate);
    return wrapped(dx);
}

OP(copy2d, "src", "dst") {
    const T s = c.tensor(0), d = c.tensor(1);
    need(s.rows() && d.rows() && s.like(d) && s.dtype() == d.dtype());
    const int64_t es = s.t.element_size();
    LAUNCH(copy2d, s.size(0), s.size(1) * es, s, s.ld() * es, d, d.ld() * es);
    return wrapped(d);
}

OP(gemm_grouped, "form", "problems", "tile") {
    const int64_t form = c.integer(0);
    need(c.integer(2, 0) == 0 && form >= 0 && form <= 2 && c.v[1] && PyList_CheckExact(c.v[1]) && kernels_int("_TILE_OVERRIDE") == 0);
    PyObject* key = PyLong_FromLong(form);
    PyObject* tile = PyDict_GetItem(kernels_item("_TILE_BY_FORM"), key);
    Py_DECREF(key);
    need(tile && PyLong_Check(tile) && PyLong_AsLong(tile) == 0);
    const int n = (int)PyList_GET_SIZE(c.v[1]);
    need(n >= 1 && n <= 8);
    mi355_gemm_problem p[8] = {};
    at::ScalarType odt = F32;
    const bool at = form == MI355_GEMM_TN, bt = form != MI355_GEMM_NT;
    for (int i = 0; i < n; ++i) {
        PyObject* q = PyList_GET_ITEM(c.v[1], i);
        need(PyTuple_CheckExact(q) && PyTuple_GET_SIZE(q) == 4);
        const T a = c.from(PyTuple_GET_ITEM(q, 0)), b = c.from(PyTuple_GET_ITEM(q, 1)), out = c.from(PyTuple_GET_ITEM(q, 2)), r = c.from(PyTuple_GET_ITEM(q, 3));
        need(a && b && out && a.rows() && b.rows() && out.rows() && a.is(BF16) && b.is(BF16));
        if (i == 0) odt = out.dtype();
        const int64_t M = a.size(at), K = a.size(!at), N = b.size(bt);
        need(b.size(!bt) == K && out.shape({M, N}) && out.dtype() == odt && (!r || (r.rows() && r.dtype() == odt && r.shape({M, N}))));
        p[i].M = M, p[i].N = N, p[i].K = K, p[i].A = a.ptr(), p[i].lda = a.ld(), p[i].B = b.ptr(), p[i].ldb = b.ld(), p[i].C = out.ptr(), p[i].ldc = out.ld(), p[i].residual = r.ptr(), p[i].ldr = r.ld();
    }
    const bool split = at && p[0].K >= kernels_int("GROUP_SPLIT_MIN_K");
    T ws;
    if (split) ws = c.workspace(c.from(PyTuple_GET_ITEM(PyList_GET_ITEM(c.v[1], 0), 0)));
    LAUNCH(gemm_bf16_grouped_ws, form, n, p, code(odt), 0, ws, split ? kernels_int("WS_BYTES") : 0L);
    Py_RETURN_NONE;
}

// ---------------------------------------------------------------------------------------------- kernels_q35.py
T reduce_parts(Call& c, const T& part) {
    const T out = c.empty(part, {part.size(1)}, F32);
    LAUNCH(reduce_rows_f32, part.size(0), part.size(1), part, out, MI355_DT_F32, 0);
    return out;
}
bool cols(const T& t, at::ScalarType s = BF16) { return t.rows() && t.is(s); }
bool heads(const T& t, int64_t H, int64_t D, int64_t hs) { return cols(t) && t.size(1) >= (H - 1) * hs + D; }

OP(zc_weight, "scale") {
    const T s = c.tensor(0);
    need(s.is(BF16) && s.contiguous());
    const T w = c.empty_like(s);
    LAUNCH(zc_weight, s.numel(), s, w);
    return wrapped(w);
}

OP(headnorm_rope_fwd, "src", "H", "D", "head_stride", "w_eff", "cos_t", "sin_t", "pos", "eps") {
    const T src = c.tensor(0), w = c.tensor(4), cos = c.maybe(5), sin = c.maybe(6), pos = c.maybe(7);
    const int64_t H = c.integer(1), D = c.integer(2), hs = c.integer(3);
    need(heads(src, H, D, hs) && w.vec(BF16, D) && (!cos || cos.dim() == 2));
    const int64_t tokens = src.size(0), R = cos ? cos.size(1) : 0;
    if (R) need(cos.is(F32) && sin && sin.is(F32) && cos.contiguous() && sin.contiguous() && sin.like(cos) && pos && pos.vec(I32, tokens));
    const T out = c.empty(src, {tokens, H * D}, BF16), rstd = c.empty(src, {tokens, H}, F32);
    LAUNCH(headnorm_rope_fwd, tokens, H, D, R, src, src.ld(), hs, w, cos, sin, pos, out, rstd, c.real(8, 1e-6));
    return tuple(out, rstd);
}

OP(headnorm_rope_bwd, "src", "H", "D", "head_stride", "w_eff", "cos_t", "sin_t", "pos", "rstd", "dout", "dsrc", "dhead_stride", "partial") {
    const T src = c.tensor(0), w = c.maybe(4), cos = c.maybe(5), sin = c.maybe(6), pos = c.maybe(7), rstd = c.maybe(8), dout = c.tensor(9), dsrc = c.tensor(10);
    const int64_t H = c.integer(1), D = c.integer(2), hs = c.integer(3), dhs = c.integer(11);
    need(heads(src, H, D, hs) && heads(dsrc, H, D, dhs) && (!cos || cos.dim() == 2));
    const int64_t tokens = src.size(0), R = cos ? cos.size(1) : 0, parts = std::max<int64_t>(1, std::min<int64_t>(c.constant("NORM_PARTS"), (tokens * H + 3) / 4));
    need(dout.is(BF16) && dout.contiguous() && dout.shape({tokens, H * D}) && (dry || slot::reduce_rows_f32.address));
    const T part = c.empty(src, {parts, D}, F32);
    LAUNCH(headnorm_rope_bwd, tokens, H, D, R, src, src.ld(), hs, w, cos, sin, pos, rstd, dout, dsrc, dsrc.ld(), dhs, part, parts);
    return wrapped(c.truth(12, false) ? part : reduce_parts(c, part));
}

OP(sigmoid_gate_fwd, "ctx", "gate", "H", "D", "gate_head_stride") {
    const T ctx = c.tensor(0), gate = c.tensor(1);
    const int64_t H = c.integer(2), D = c.integer(3), ghs = c.integer(4);
    need(heads(gate, H, D, ghs) && ctx.dim() == 2 && ctx.is(BF16) && ctx.contiguous() && ctx.size(1) == H * D && ctx.size(0) == gate.size(0));
    const T out = c.empty_like(ctx);
    LAUNCH(sigmoid_gate_fwd, ctx.size(0), H, D, ctx, gate, gate.ld(), ghs, out);
    return wrapped(out);
}

OP(sigmoid_gate_bwd, "ctx", "gate", "H", "D", "gate_head_stride", "dout", "dgate", "dgate_head_stride") {
    const T ctx = c.tensor(0), gate = c.tensor(1), dout = c.tensor(5), dgate = c.tensor(6);
    const int64_t H = c.integer(2), D = c.integer(3), ghs = c.integer(4), dghs = c.integer(7);
    need(heads(gate, H, D, ghs) && heads(dgate, H, D, dghs) && ctx.dim() >= 1 && dout.is(BF16) && dout.contiguous() && dout.like(ctx));
    const T dctx = c.empty_like(ctx);
    LAUNCH(sigmoid_gate_bwd, ctx.size(0), H, D, ctx, gate, gate.ld(), ghs, dout, dctx, dgate, dgate.ld(), dghs);
    return wrapped(dctx);
}

OP(attn_generic_fwd, "q", "k", "v", "B", "S", "Hq", "Hkv", "D", "key_mask", "scale") {
    const T q = c.tensor(0), k = c.tensor(1), v = c.tensor(2), mask = c.maybe(8);
    const int64_t B = c.integer(3), S = c.integer(4), Hq = c.integer(5), Hkv = c.integer(6), D = c.integer(7);
    need(D > 0 && attn_operand(q, B * S, Hq * D) && attn_operand(k, B * S, Hkv * D) && attn_operand(v, B * S, Hkv * D) && (!mask || (mask.is(U8) && mask.contiguous() && mask.shape({B, S}))));
    const double scale = c.given(9) ? c.real(9) : std::pow((double)D, -0.5);
    const T o = c.empty(q, {B * S, Hq * D}, BF16), lse = c.empty(q, {B, Hq, S}, F32);
    LAUNCH(attn_generic_fwd, B, S, Hq, Hkv, D, q, q.ld(), k, k.ld(), v, v.ld(), o, o.ld(), lse, mask, scale);
    return tuple(o, lse);
}

OP(attn_generic_bwd, "q", "k", "v", "o", "do", "lse", "B", "S", "Hq", "Hkv", "D", "dq", "dk", "dv", "key_mask", "scale") {
    const T q = c.tensor(0), k = c.tensor(1), v = c.tensor(2), o = c.tensor(3), dO = c.tensor(4), lse = c.tensor(5), dq = c.tensor(11), dk = c.tensor(12), dv = c.tensor(13), mask = c.maybe(14);
    const int64_t B = c.integer(6), S = c.integer(7), Hq = c.integer(8), Hkv = c.integer(9), D = c.integer(10);
    need(D > 0);
    for (const T* t : {&q, &o, &dO, &dq}) need(attn_operand(*t, B * S, Hq * D));
    for (const T* t : {&k, &v, &dk, &dv}) need(attn_operand(*t, B * S, Hkv * D));
    need(lse.is(F32) && lse.contiguous() && lse.shape({B, Hq, S}));
    const double scale = c.given(15) ? c.real(15) : std::pow((double)D, -0.5);
    const T delta = c.empty_like(lse);
    LAUNCH(attn_generic_bwd, B, S, Hq, Hkv, D, q, q.ld(), k, k.ld(), v, v.ld(), o, o.ld(), dO, dO.ld(), lse, delta, dq, dq.ld(), dk, dk.ld(), dv, dv.ld(), mask, scale);
    Py_RETURN_NONE;
}

OP(gdn_gates_fwd, "b_lin", "a_lin", "log_A", "dt_bias") {
    const T b = c.tensor(0), a = c.tensor(1), A = c.tensor(2), dt = c.tensor(3);
    need(cols(b) && cols(a) && a.like(b) && a.ld() == b.ld());
    const int64_t tokens = b.size(0), H = b.size(1);
    need(A.is(F32) && dt.is(BF16) && A.numel() == H && dt.numel() == H);
    const T beta = c.empty(b, {tokens, H}, F32), alpha = c.empty_like(beta);
    LAUNCH(gdn_gates_fwd, tokens, H, b, a, b.ld(), A, dt, beta, alpha);
    return tuple(beta, alpha);
}

OP(gdn_gates_bwd, "b_lin", "a_lin", "log_A", "dt_bias", "dbeta", "dalpha", "db_lin", "da_lin", "partial") {
    const T b = c.tensor(0), a = c.tensor(1), A = c.tensor(2), dt = c.tensor(3), dbeta = c.tensor(4), dalpha = c.tensor(5), db = c.tensor(6), da = c.tensor(7);
    need(b.dim() == 2 && cols(db) && cols(da));
    const int64_t tokens = b.size(0), H = b.size(1), parts = std::max<int64_t>(1, std::min<int64_t>(256, (tokens * H + 255) / 256));
    need(db.ld() == da.ld() && db.shape({tokens, H}) && da.shape({tokens, H}));
    for (const T* t : {&dbeta, &dalpha}) need(t->is(F32) && t->contiguous() && t->shape({tokens, H}));
    need(dry || slot::reduce_rows_f32.address);
    const T part = c.empty(b, {parts, 2 * H}, F32);
    LAUNCH(gdn_gates_bwd, tokens, H, b, a, b.ld(), A, dt, dbeta, dalpha, db, da, db.ld(), part, parts);
    if (c.truth(8, false)) return tuple(T{part.t.narrow(1, 0, H)}, T{part.t.narrow(1, H, H)});
    const T both = reduce_parts(c, part);
    return tuple(T{both.t.narrow(0, 0, H)}, T{both.t.narrow(0, H, H)});
}

OP(causal_conv_silu_fwd, "x", "w", "B", "S") {
    const T x = c.tensor(0), w = c.tensor(1);
    const int64_t B = c.integer(2), S = c.integer(3);
    need(cols(x) && w.dim() >= 1 && x.size(0) == B * S && w.is(BF16) && w.contiguous() && w.size(0) == x.size(1) && w.numel() == x.size(1) * w.size(w.dim() - 1));
    const T y = c.empty(x, {B * S, x.size(1)}, BF16);
    LAUNCH(causal_conv_silu_fwd, B, S, x.size(1), w.size(w.dim() - 1), x, x.ld(), w, y);
    return wrapped(y);
}

OP(causal_conv_silu_bwd, "x", "w", "dy", "dx", "B", "S", "partial") {
    const T x = c.tensor(0), w = c.tensor(1), dy = c.tensor(2), dx = c.tensor(3);
    const int64_t B = c.integer(4), S = c.integer(5), chunk = c.constant("CONV_TOKEN_CHUNK");
    need(chunk > 0 && cols(x) && cols(dx) && w.dim() >= 1 && dy.is(BF16) && dy.contiguous() && dy.shape({B * S, x.size(1)}) && dx.shape({B * S, x.size(1)}) && (dry || slot::reduce_rows_f32.address));
    const int64_t C = x.size(1), ks = w.size(w.dim() - 1);
    const void* mine = dx.t.storage().data();  // only a gradient that overwrites its operands needs scratch
    const T ws = mine == x.t.storage().data() || mine == dy.t.storage().data() ? c.empty(x, {B * S, C}, BF16) : T{};
    const T part = c.empty(x, {B * ((S + chunk - 1) / chunk), C * ks}, F32);
    LAUNCH(causal_conv_silu_bwd, B, S, C, ks, x, x.ld(), w, dy, ws, dx, dx.ld(), part, chunk);
    return wrapped(c.truth(6, false) ? part : reduce_parts(c, part));
}

OP(l2norm_fwd, "x", "H", "D") {
    const T x = c.tensor(0);
    const int64_t H = c.integer(1), D = c.integer(2);
    need(cols(x) && x.size(1) == H * D);
    const T y = c.empty(x, {x.size(0), H * D}, BF16);
    LAUNCH(l2norm_fwd, x.size(0), H, D, x, x.ld(), y);
    return wrapped(y);
}

OP(l2norm_bwd, "x", "dy", "dx", "H", "D") {
    const T x = c.tensor(0), dy = c.tensor(1), dx = c.tensor(2);
    const int64_t H = c.integer(3), D = c.integer(4);
    need(cols(x) && cols(dx) && dy.is(BF16) && dy.contiguous() && dy.shape({x.size(0), H * D}) && dx.like(x));
    LAUNCH(l2norm_bwd, x.size(0), H, D, x, x.ld(), dy, dx, dx.ld());
    Py_RETURN_NONE;
}

OP(gated_rmsnorm_fwd, "o", "w_f32", "gate", "H", "D", "eps") {
    const T o = c.tensor(0), w = c.tensor(1), gate = c.tensor(2);
    const int64_t H = c.integer(3), D = c.integer(4);
    need(cols(gate) && o.dim() == 2 && o.is(BF16) && o.contiguous() && o.size(1) == H * D && gate.like(o) && w.is(F32) && w.numel() == D);
    const T out = c.empty_like(o), rstd = c.empty(o, {o.size(0), H}, F32);
    LAUNCH(gated_rmsnorm_fwd, o.size(0), H, D, o, w, gate, gate.ld(), out, rstd, c.real(5, 1e-6));
    return tuple(out, rstd);
}

OP(gated_rmsnorm_bwd, "o", "w_f32", "gate", "rstd", "dout", "dgate", "H", "D", "partial") {
    const T o = c.tensor(0), w = c.tensor(1), gate = c.tensor(2), rstd = c.tensor(3), dout = c.tensor(4), dgate = c.tensor(5);
    const int64_t H = c.integer(6), D = c.integer(7);
    need(cols(dgate) && o.dim() == 2 && gate.dim() >= 1 && dout.is(BF16) && dout.contiguous() && dout.like(o) && dgate.like(o) && (dry || slot::reduce_rows_f32.address));
    const int64_t parts = std::max<int64_t>(1, std::min<int64_t>(c.constant("NORM_PARTS"), (o.size(0) * H + 3) / 4));
    const T d_o = c.empty_like(o), part = c.empty(o, {parts, D}, F32);
    LAUNCH(gated_rmsnorm_bwd, o.size(0), H, D, o, w, gate, gate.ld(), rstd, dout, d_o, dgate, dgate.ld(), part, parts);
    return tuple(d_o, c.truth(8, false) ? part : reduce_parts(c, part));
}

// ---------------------------------------------------------------------------------------------- ops_decode.py, kernels_seq.py
T stream_product(Call& c, const T& x, const T& w, const T& residual) {  // ops_decode.gemv of at most eight rows
    const int64_t M = x.size(0);
    need(M <= 8 && x.is(BF16) && w.is(BF16) && x.rows() && w.rows() && x.size(1) == w.size(1));
    const T y = c.empty(x, {M, w.size(0)}, BF16);
    LAUNCH(gemv_bf16, M, w.size(0), w.size(1), x, x.ld(), w, w.ld(), y, y.ld(), residual, residual.ld());
    return y;
}
OP(gemv, "x2d", "w", "residual") {
    const T x = c.tensor(0), w = c.tensor(1), residual = c.maybe(2);
    need(x.dim() == 2 && (!residual || residual.dim() >= 1));
    return wrapped(stream_product(c, x, w, residual));
}

OP(bgemm, "a", "b", "c", "M", "N", "Kd", "batch", "lda", "a_bs", "sbn", "sbk", "b_bs", "ldc", "c_bs", "grp_offs", "a_rows", "a_div", "c_rows", "row_scale", "epi", "mfma", "bias", "limit", "n_out") {
    const T a = c.tensor(0), b = c.tensor(1), out = c.tensor(2), grp = c.maybe(14), ar = c.maybe(15), cr = c.maybe(17), rs = c.maybe(18), bias = c.maybe(21);
    const int64_t N = c.integer(4);
    need(a.dim() >= 1 && b.dim() >= 1 && out.dim() >= 1 && (!bias || bias.vec(F32, N)));
    const bool mfma = c.given(20) ? c.truth(20, false) : a.is(BF16) && b.is(BF16);
    LAUNCH(bgemm, c.integer(6, 1), c.integer(3), N, c.integer(5), a, a.code(), c.given(7) ? c.integer(7) : a.ld(), c.integer(8, 0), b, b.code(), c.given(9) ? c.integer(9) : b.ld(), c.integer(10, 1),
           c.integer(11, 0), out, out.code(), c.given(12) ? c.integer(12) : out.ld(), c.integer(13, 0), grp, ar, c.integer(16, 1), cr, rs, c.integer(19, 0), (int)mfma, bias, c.real(22, 0.0), c.integer(23, 0));
    return wrapped(out);
}

OP(linear, "x", "w", "out_dtype", "bias") {
    const T x = c.tensor(0), w = c.tensor(1), bias = c.maybe(3);
    need(x.rows() && w.dim() == 2 && w.is(BF16) && w.size(1) == x.size(1) && w.t.strides()[1] == 1);
    const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
    const at::ScalarType od = c.dtype(2, x.dtype());
    need((x.is(BF16) || x.is(F32)) && (od == BF16 || od == F32));
    if (x.is(BF16) && K % 8 == 0 && x.ld() % 8 == 0 && w.ld() % 8 == 0 && x.addr() % 16 == 0 && w.addr() % 16 == 0) {
        if (M <= 8 && od == BF16 && !bias) return wrapped(stream_product(c, x, w, T{}));
        if (M <= 8 && od == F32 && (!bias || bias.vec(F32, N))) {
            const T out = c.empty(x, {M, N}, F32);
            LAUNCH(gemv_bf16_f32out, M, N, K, x, x.ld(), w, w.ld(), out, out.ld(), bias);
            return wrapped(out);
        }
        if (M > 8) return wrapped(product(c, MI355_GEMM_NT, x, w, T{}, od, bias, T{}, MI355_EPI_NONE, true));
    }
    need(!bias || bias.vec(F32, N));
    const T out = c.empty(x, {M, N}, od);
    LAUNCH(bgemm, 1, M, N, K, x, x.code(), x.ld(), 0, w, w.code(), w.ld(), 1, 0, out, out.code(), out.ld(), 0, T{}, T{}, 1, T{}, T{}, 0, (int)x.is(BF16), bias, 0.0, 0);
    return wrapped(out);
}

OP(hyper_mix, "x", "S", "y", "parts", "y_scale", "mix", "put", "read", "rows", "x_out", "want_u", "norm", "eps", "out_dtype") {
    const T x = c.tensor(0), y = c.maybe(2), mix = c.maybe(5), put = c.maybe(6), read = c.maybe(7), rows = c.maybe(8), norm = c.maybe(11);
    const bool make = c.v[9] == Py_True;
    T x_out = make ? T{} : c.maybe(9);
    const int64_t S = c.integer(1), parts = c.integer(3, 1);
    need((x.dim() == 2 || (x.dim() == 3 && x.size(1) == S)) && x.is(F32) && x.t.strides().back() == 1);
    const int64_t n = x.size(0), width = x.size(x.dim() - 1), tokens = rows ? rows.numel() : n;
    need(!rows || (rows.is(I64) && rows.contiguous()));
    need(!y || (y.rows() && y.shape({n * parts, width}) && mix && put));
    need(mix.vec_or_none(F32, S * S) && put.vec_or_none(F32, S) && read.vec_or_none(F32, S) && norm.vec_or_none(F32, width));
    need(!x_out || (x_out.is(F32) && x_out.contiguous() && x_out.shape({tokens, S, width})));
    const double scale = c.real(4, 1.0), eps = c.real(12, 0.0);
    const int yc = y.code();
    const at::ScalarType od = c.dtype(13, F32);
    if (make) x_out = c.empty(x, {tokens, S, width}, F32);
    const T out = norm ? c.empty(x, {tokens, width}, od) : T{}, u = c.truth(10, false) ? c.empty(x, {tokens, width}, F32) : T{};
    LAUNCH(hyper_mix, tokens, width, S, x, x.ld(), x.dim() == 3 ? x.t.strides()[1] : 0, y, yc, y.ld(), parts, scale, mix, put, read, rows, x_out, u, norm, eps, out, out.code());
    return tuple(x_out, out, u);
}

bool ints(const T& t, int64_t n = 0) { return t.is(I32) && t.contiguous() && t.numel() >= n; }

// kernels_seq.attn_key_splits
int64_t key_splits(int64_t n_seq, int64_t head_tiles, int64_t max_new, int64_t hm, int64_t max_keys, int64_t per_split) {
    const int64_t tiles = n_seq * head_tiles * ((max_new * hm + 127) / 128);
    if (max_keys <= 2 * per_split || tiles >= 128) return 1;
    return std::max<int64_t>(1, std::min<int64_t>({(max_keys + per_split - 1) / per_split, 32, 256 / tiles}));
}

OP(latent_attn, "q", "k1", "k2", "v", "out", "H", "hm", "D1", "D2", "DV", "q_hs", "k1_hs", "v_hs", "o_hs", "desc", "max_new", "scale", "max_keys", "kv_rep", "window", "keep_first", "softcap", "sink", "pool",
   "pooled", "pool_row0", "chunk", "sig_bias", "slope", "gate") {
    const T q = c.tensor(0), k1 = c.tensor(1), k2 = c.maybe(2), v = c.tensor(3), out = c.tensor(4), sink = c.maybe(22), sig = c.maybe(27), slope = c.maybe(28), gate = c.maybe(29);
    const int64_t H = c.integer(5), hm = c.integer(6), D1 = c.integer(7), D2 = c.integer(8), DV = c.integer(9), max_new = c.integer(15), max_keys = c.integer(17, 0), window = c.integer(19, 0),
                  keep = c.integer(20, 0), chunk = c.integer(26, 0);
    need(c.integer(23, 0) == 0 && H > 0 && hm > 0 && max_new > 0 && max_keys >= 0 && window >= 0 && chunk >= 0 && keep >= 0 && DV > 0);  // (pooled rows: Python)
    need(q.rows() && k1.rows() && v.rows() && out.rows() && (!k2 || k2.dim() >= 1));
    need(slope.vec_or_none(F32, H) && sig.vec_or_none(F32, H) && sink.vec_or_none(F32, H) && (!gate || (gate.rows() && gate.is(F32) && gate.shape({q.size(0), H * DV}))));
    need(q.is(F32) && k1.dtype() == v.dtype() && (out.dtype() == v.dtype() || out.is(F32)) && (!k2 || k2.dtype() == v.dtype()));
    PyObject* desc = c.v[14];
    need(desc && PyTuple_CheckExact(desc) && PyTuple_GET_SIZE(desc) == 6);
    T d[6];
    for (int i = 0; i < 6; ++i) d[i] = c.from(PyTuple_GET_ITEM(desc, i)), need(bool(d[i]));
    const int64_t n_seq = d[0].numel();
    for (const T& t : d) need(ints(t, n_seq));
    need(n_seq > 0);
    const bool mfma = v.is(BF16);
    int64_t splits = 1;
    T ws;
    const int64_t reach = std::min(window ? window : chunk, chunk ? chunk : window);
    if (mfma && D1 + D2 <= 320 && DV <= 256 && max_keys) {
        const int64_t head_tiles = (H + hm - 1) / hm, tile_tokens = std::min(max_new, (128 + hm - 1) / hm);
        if (reach && reach < max_keys) splits = key_splits(n_seq, head_tiles, max_new, hm, std::min(max_keys, keep + reach + tile_tokens - 1), 128);
        else splits = key_splits(n_seq, head_tiles, max_new, hm, max_keys, 256);
        if (splits > 1) {
            const int64_t dvp = DV <= 32 ? 32 : DV <= 64 ? 64 : DV <= 128 ? 128 : 256;
            ws = c.empty(v, {n_seq * head_tiles * ((max_new * hm + 127) / 128) * splits * 128 * (2 + dvp)}, F32);
        }
    }
    const double softcap = c.given(21) ? c.real(21) : 0.0;
    LAUNCH(latent_attn, n_seq, max_new, H, hm, D1, D2, DV, q, q.ld(), c.integer(10), k1, k1.ld(), c.integer(11), k2, k2.ld(), v, v.ld(), c.integer(12), out, out.ld(), c.integer(13), v.code(), d[0], d[1], d[2],
           d[3], d[4], d[5], c.real(16), (int)mfma, splits, ws, ws ? ws.numel() : 0, c.integer(18, 1), window, keep, softcap, sink, 0, T{}, T{}, 0, c.maybe(25), chunk, sig, out.code(), slope, gate, gate.ld());
    return wrapped(out);
}

OP(qkv_rows_append, "src", "H", "G", "d", "dv", "bias", "qw", "kw", "eps", "qscale", "dims", "layout", "freq", "pos", "dst_row", "cache2d", "q_temp", "vmix", "lam", "v_heads", "unit_norm", "rot_amp", "tie_v") {
    const T src = c.tensor(0), bias = c.maybe(5), qw = c.maybe(6), kw = c.maybe(7), qscale = c.maybe(9), freq = c.maybe(12), pos = c.tensor(13), dst = c.tensor(14), cache = c.tensor(15), vmix = c.maybe(17);
    const int64_t H = c.integer(1), G = c.integer(2), d = c.integer(3), dv = c.integer(4), dims = c.integer(10), GV = c.given(19) && c.integer(19) ? c.integer(19) : G;
    const bool tie = c.truth(22, false);
    need(!c.given(16) && src.rows() && cache.rows() && dims >= 0);  // (query temperatures: Python)
    const int64_t tokens = src.size(0), n_in = (H + G) * d + (tie ? 0 : GV * dv);
    need(!vmix || (vmix.rows() && vmix.is(F32) && vmix.shape({tokens, GV * dv})));
    need(src.size(1) == n_in && cache.size(1) == G * d + GV * dv);
    const auto vec = [](const T& t, int64_t n) { return !t || (t.is(F32) && t.contiguous() && t.numel() >= n); };
    need(vec(bias, n_in) && vec(qw, d) && vec(kw, d) && vec(qscale, H) && vec(freq, dims / 2) && ints(pos, tokens) && ints(dst, tokens));
    const int sc = src.code(), cc = cache.code();
    const T q = c.empty(src, {tokens, H * d}, F32);
    LAUNCH(qkv_rows_append, tokens, H, G, d, dv, src, sc, src.ld(), bias, qw, kw, c.real(8), qscale, dims, c.integer(11), freq, pos, dst, q, q.ld(), cache, cc, cache.ld(), 0.0, 0, vmix, vmix.ld(), c.real(18, 0.0),
           GV, (int)c.truth(20, false), c.real(21, 1.0), (int)tie);
    return wrapped(q);
}

OP(group_rmsnorm_sum, "x", "groups", "eps", "y1", "y2", "parts", "x_out", "norm_a", "norm_b") {
    const T x = c.tensor(0), y1 = c.maybe(3), y2 = c.maybe(4);
    const int64_t parts = c.integer(5, 1);
    need(x.rows() && x.is(F32) && x.contiguous());
    const int64_t tokens = x.size(0), width = x.size(1);
    need((!y1 || (y1.rows() && y1.shape({tokens, width}))) && (!y2 || (y2.rows() && y2.shape({tokens * parts, width}))));
    const bool make = c.v[6] == Py_True;
    T x_out = make ? T{} : c.maybe(6);
    need(!x_out || (x_out.is(F32) && x_out.contiguous() && x_out.like(x)));  // (anything else: Python passes the pointer on)
    struct Norm {
        T w, o, o32;
        bool given = false, want = false, same = false;
        at::ScalarType s = F32;
    } norm[2];
    for (int i = 0; i < 2; ++i) {
        PyObject* o = c.v[7 + i];
        if (!o || o == Py_None) continue;
        need(PyTuple_CheckExact(o) && PyTuple_GET_SIZE(o) == 3 && PyBool_Check(PyTuple_GET_ITEM(o, 2)));
        Norm& m = norm[i];
        m.w = c.from(PyTuple_GET_ITEM(o, 0));
        need(bool(m.w) && m.w.vec(F32, width));
        PyObject* s = PyTuple_GET_ITEM(o, 1);
        need(s == Py_None || THPDtype_Check(s));
        m.given = s != Py_None, m.want = PyTuple_GET_ITEM(o, 2) == Py_True;
        if (m.given) m.s = reinterpret_cast<THPDtype*>(s)->scalar_type, need(m.s == BF16 || m.s == F32);
        m.same = m.given && m.s == F32 && m.want;
    }
    const int c1 = y1.code(), c2 = y2.code();
    const int64_t groups = c.integer(1);
    const double eps = c.real(2);
    if (make) x_out = c.empty_like(x);
    for (Norm& m : norm) {
        if (m.given) m.o = c.empty(x, {tokens, width}, m.s);
        if (m.want) m.o32 = m.same ? m.o : c.empty(x, {tokens, width}, F32);
    }
    LAUNCH(group_rmsnorm_sum, tokens, width, x, y1, c1, y1.ld(), y2, c2, y2.ld(), parts, x_out, groups, eps, norm[0].w, norm[0].o, norm[0].o.code(), norm[0].same ? T{} : norm[0].o32, norm[1].w, norm[1].o,
           norm[1].o.code(), norm[1].same ? T{} : norm[1].o32);
    PyObject* pair[2];
    for (int i = 0; i < 2; ++i) {
        PyObject* o = wrapped(norm[i].o);
        PyObject* o32 = norm[i].same ? Py_NewRef(o) : wrapped(norm[i].o32);  // (one object where they are one tensor)
        pair[i] = PyTuple_New(2);
        PyTuple_SET_ITEM(pair[i], 0, o);
        PyTuple_SET_ITEM(pair[i], 1, o32);
    }
    PyObject* out = PyTuple_New(3);
    PyTuple_SET_ITEM(out, 0, make || !c.given(6) ? wrapped(x_out) : Py_NewRef(c.v[6]));
    PyTuple_SET_ITEM(out, 1, pair[0]);
    PyTuple_SET_ITEM(out, 2, pair[1]);
    return out;
}

OP(ragged_conv, "x", "w", "state", "row_seq", "seq_off", "slot", "act", "residual", "out_dtype", "bias") {
    const T x = c.tensor(0), w = c.tensor(1), state = c.maybe(2), row_seq = c.tensor(3), seq_off = c.tensor(4), slot_ = c.tensor(5), bias = c.maybe(9);
    need(x.rows() && w.dim() == 2 && w.is(F32) && w.contiguous() && w.size(0) == x.size(1) && bias.vec_or_none(F32, x.size(1)));
    const int64_t tokens = x.size(0), C = x.size(1), taps = w.size(1), n_seq = slot_.numel();
    need(taps <= 1 || (state && state.dim() == 3 && state.is(F32) && state.contiguous() && state.size(1) == taps - 1 && state.size(2) == C));
    need(ints(row_seq, tokens) && ints(seq_off, n_seq + 1) && ints(slot_));
    const int xc = x.code();
    const T y = c.empty(x, {tokens, C}, c.dtype(8, x.dtype()));
    LAUNCH(ragged_conv, tokens, n_seq, C, taps, x, xc, x.ld(), w, row_seq, seq_off, slot_, state, (int)c.truth(6, false), (int)c.truth(7, false), y, y.code(), y.ld(), bias);
    return wrapped(y);
}

OP(gated_headnorm, "o", "w", "gate", "H", "D", "eps", "out_dtype") {
    const T o = c.tensor(0), w = c.tensor(1), gate = c.tensor(2);
    const int64_t H = c.integer(3), D = c.integer(4);
    need(gate.rows() && o.dim() == 2 && o.is(F32) && o.contiguous() && o.size(1) == H * D && gate.like(o) && w.is(F32) && w.numel() == D && c.given(6));
    const int gc = gate.code();
    const double eps = c.real(5);
    const T out = c.empty(o, {o.size(0), o.size(1)}, c.dtype(6, F32));
    LAUNCH(gated_headnorm, o.size(0), H, D, o, w, gate, gc, gate.ld(), eps, out, out.code(), out.ld());
    return wrapped(out);
}

OP(glu_rows, "x", "kind", "limit", "out_dtype") {
    const T x = c.tensor(0);
    need(x.rows());
    const int64_t F = x.size(1) / 2, kind = c.integer(1);
    const double limit = c.real(2, 0.0);
    const int xc = x.code();
    const T out = c.empty(x, {x.size(0), F}, c.dtype(3, x.dtype()));
    LAUNCH(glu_rows, x.size(0), F, x, xc, x.ld(), kind, limit, out, out.code(), out.ld());
    return wrapped(out);
}

OP(add_layernorm, "x", "w", "b", "eps", "alpha", "y", "parts", "cast_dtype") {
    const T x = c.tensor(0), w = c.tensor(1), b = c.tensor(2), y = c.maybe(5);
    const int64_t parts = c.integer(6, 1);
    need(x.rows() && x.is(F32) && x.contiguous() && w.is(F32) && b.is(F32));
    const int64_t tokens = x.size(0), width = x.size(1);
    need(w.numel() == width && b.numel() == width && (!y || (y.rows() && y.shape({tokens * parts, width}))));
    const int yc = y.code();
    const double eps = c.real(3), alpha = c.real(4, 1.0);
    const bool cast = c.given(7), own = cast && c.dtype(7, F32) != F32;
    const T out = c.empty_like(x), low = own ? c.empty(x, {tokens, width}, c.dtype(7, F32)) : T{};
    LAUNCH(add_layernorm_fwd, tokens, width, x, alpha, y, yc, y.ld(), parts, w, b, eps, out, low, low.code());
    if (own || !cast) return tuple(out, low);
    PyObject* o = wrapped(out);
    PyObject* pair = PyTuple_Pack(2, o, o);
    Py_DECREF(o);
    return pair;
}

OP(rmsnorm_rows, "x", "w", "eps", "out_dtype") {
    const T x = c.tensor(0), w = c.tensor(1);
    need(x.rows() && w.is(F32) && w.numel() == x.size(1));
    const int xc = x.code();
    const double eps = c.real(2);
    const T out = c.empty(x, {x.size(0), x.size(1)}, c.dtype(3, x.dtype()));
    LAUNCH(rmsnorm_rows, x.size(0), x.size(1), x, xc, x.ld(), w, eps, out, out.code(), out.ld());
    return wrapped(out);
}

OP(latent_kv_append, "src", "rank", "rot", "w", "eps", "pos", "dst_row", "freq", "dims", "cache2d", "layout") {
    const T src = c.tensor(0), w = c.tensor(3), pos = c.tensor(5), dst = c.tensor(6), freq = c.maybe(7), cache = c.tensor(9);
    const int64_t rank = c.integer(1), rot = c.integer(2), dims = c.integer(8);
    need(src.rows() && cache.rows() && ints(pos, src.size(0)) && ints(dst, src.size(0)) && src.size(1) == rank + rot && cache.size(1) == rank + rot && w.is(F32) && w.numel() == rank);
    need(dims >= 0 && (!dims || (freq && freq.is(F32) && freq.numel() >= dims / 2)));
    LAUNCH(latent_kv_append, src.size(0), rank, rot, src, src.code(), src.ld(), w, c.real(4), pos, dst, freq, dims, c.integer(10, 0), cache, cache.code(), cache.ld());
    Py_RETURN_NONE;
}

OP(rope_heads, "src", "H", "n", "src_hs", "src_off", "dst", "dst_hs", "dst_off", "rot_start", "dims", "freq", "pos", "layout") {
    const T src = c.tensor(0), dst = c.tensor(5), freq = c.maybe(10), pos = c.tensor(11);
    const int64_t H = c.integer(1), n = c.integer(2), shs = c.integer(3), so = c.integer(4), dhs = c.integer(6), dof = c.integer(7);
    need(src.rows() && dst.rows() && dst.is(F32) && dst.size(0) == src.size(0) && ints(pos, src.size(0)));
    need(src.size(1) >= (H - 1) * shs + so + n && dst.size(1) >= (H - 1) * dhs + dof + n);
    LAUNCH(rope_heads, src.size(0), H, n, src, src.code(), src.ld(), shs, so, dst, dst.ld(), dhs, dof, c.integer(8), c.integer(9), c.integer(12, 0), freq, pos);
    return wrapped(dst);
}

OP(gla, "q", "k", "v", "z", "zbias", "inv_tau", "qscale", "seq_off", "slot", "state", "H", "dk", "dv", "head_decay", "kscale", "max_new", "min_new") {
    need(!c.given(13));  // (a fixed decay: Python, which may take chunks)
    const T q = c.tensor(0), k = c.tensor(1), v = c.tensor(2), z = c.tensor(3), zb = c.tensor(4), off = c.tensor(7), slot_ = c.tensor(8), state = c.tensor(9);
    const int64_t H = c.integer(10), dk = c.integer(11), dv = c.integer(12);
    for (const T* t : {&q, &k, &z}) need(t->rows() && t->size(1) == H * dk && t->size(0) == q.size(0));
    need(v.rows() && v.size(1) == H * dv && v.size(0) == q.size(0) && k.dtype() == q.dtype() && v.dtype() == q.dtype());
    const int64_t n_seq = slot_.numel();
    need(ints(off, n_seq + 1) && ints(slot_) && state.dim() == 4 && state.is(F32) && state.contiguous() && state.size(1) == H && state.size(2) == dk && state.size(3) == dv && zb.is(F32) && zb.numel() == H * dk);
    const int qc = q.code(), zc = z.code();
    const T o = c.empty(q, {q.size(0), H * dv}, F32);
    LAUNCH(gla_fwd, n_seq, off, slot_, H, dk, dv, q, k, v, z, qc, zc, qc, q.ld(), k.ld(), v.ld(), z.ld(), zb, c.real(5), c.real(6), T{}, c.real(14, 1.0), state, o);
    return wrapped(o);
}

OP(router_logits, "x32", "w") {
    const T x = c.tensor(0), w = c.tensor(1);
    need(x.rows() && x.is(F32) && w.is(BF16) && w.rows() && w.size(1) == x.size(1));
    const T out = c.empty(x, {x.size(0), w.size(0)}, F32);
    LAUNCH(router_logits, x.size(0), w.size(0), w.size(1), x, x.ld(), w, w.ld(), out);
    return wrapped(out);
}

OP(moe_route, "logits", "correction", "top", "groups", "keep", "scale", "softmax") {
    const T logits = c.tensor(0), corr = c.maybe(1);
    need(logits.dim() == 2 && logits.is(F32) && logits.contiguous() && (!corr || (corr.is(F32) && corr.numel() == logits.size(1))) && (!c.v[6] || PyBool_Check(c.v[6])));
    const int64_t tokens = logits.size(0), E = logits.size(1), top = c.integer(2);
    need(top > 0);
    const T ids = c.empty(logits, {tokens, top}, I32), wts = c.empty(logits, {tokens, top}, F32);
    LAUNCH(moe_route, tokens, E, top, c.integer(3), c.integer(4), logits, corr, c.real(5), (int)c.truth(6, false), ids, wts);
    return tuple(ids, wts);
}

OP(moe_dispatch, "ids", "E") {
    const T ids = c.tensor(0);
    const int64_t E = c.integer(1);
    need(ints(ids) && E > 0);
    const T offs = c.empty(ids, {E + 1}, I32), perm = c.empty(ids, {ids.numel()}, I32);
    LAUNCH(moe_dispatch, ids.numel(), E, ids, offs, perm);
    return tuple(offs, perm);
}

OP(moe_choose, "x32", "w", "correction", "top", "groups", "keep", "scale", "softmax") {
    const T x = c.tensor(0), w = c.tensor(1), corr = c.maybe(2);
    need(x.rows() && x.is(F32) && w.is(BF16) && w.rows() && w.size(1) == x.size(1) && (!corr || (corr.is(F32) && corr.numel() == w.size(0))) && (!c.v[7] || PyBool_Check(c.v[7])) && moe_choose_takes);
    const int64_t tokens = x.size(0), E = w.size(0), K = w.size(1), top = c.integer(3);
    need(tokens > 0 && E > 0 && top > 0 && top <= E && E <= 512 && K <= 16384 && (dry || (slot::moe_choose.address && slot::router_logits.address && slot::moe_route.address && slot::moe_dispatch.address)));
    const bool one = moe_choose_takes(tokens, E, K, top);
    const T logits = one ? T{} : c.empty(x, {tokens, E}, F32), ids = c.empty(x, {tokens, top}, I32), wts = c.empty(x, {tokens, top}, F32), offs = c.empty(x, {E + 1}, I32), perm = c.empty(x, {tokens * top}, I32);
    if (one) {
        LAUNCH(moe_choose, tokens, E, K, top, c.integer(4), c.integer(5), x, x.ld(), w, w.ld(), corr, c.real(6), (int)c.truth(7, false), ids, wts, offs, perm);
    } else {
        LAUNCH(router_logits, tokens, E, K, x, x.ld(), w, w.ld(), logits);
        LAUNCH(moe_route, tokens, E, top, c.integer(4), c.integer(5), logits, corr, c.real(6), (int)c.truth(7, false), ids, wts);
        LAUNCH(moe_dispatch, tokens * top, E, ids, offs, perm);
    }
    return tuple(ids, wts, offs, perm);
}

OP(unary_rows, "x", "kind", "gate", "group", "out_dtype", "limit") {
    const T x = c.tensor(0), gate = c.maybe(2);
    const int64_t kind = c.integer(1), group = c.integer(3, 1);
    need(x.rows() && !gate && kind != 2);  // (the gated kind: Python)
    const int xc = x.code();
    const double limit = c.real(5, 0.0);
    const T out = c.empty(x, {x.size(0), x.size(1)}, c.dtype(4, x.dtype()));
    LAUNCH(unary_rows, x.size(0), x.size(1), x, xc, x.ld(), kind, T{}, 0, 0, group, limit, out, out.code(), out.ld());
    return wrapped(out);
}

OP(embed_hash, "tok", "prev", "table", "scale", "bigram", "buckets", "mul_prev", "mul_cur", "out") {
    const T tok = c.tensor(0), prev = c.maybe(1), table = c.tensor(2), bigram = c.maybe(4);
    T out = c.maybe(8);
    const int64_t tokens = tok.numel(), buckets = c.integer(5, 0);
    need(ints(tok) && table.dim() == 2 && table.is(BF16) && table.contiguous());
    need(!bigram || (prev && ints(prev, tokens) && bigram.is(BF16) && bigram.contiguous() && bigram.shape({buckets + 1, table.size(1)})));
    const double scale = c.real(3);
    if (!out) out = c.empty(table, {tokens, table.size(1)}, F32);
    need(out.is(F32) && out.contiguous() && out.shape({tokens, table.size(1)}));
    LAUNCH(embed_hash_fwd, tokens, table.size(1), table.size(0), tok, prev, table, scale, bigram, buckets, c.integer(6, 0), c.integer(7, 0), out);
    return wrapped(out);
}

// ---------------------------------------------------------------------------------------------- the operators as callables
// What a function can do besides being called an operator can too: it is pickled and copied by its module and name, weakly referenced, bound where it is a class's attribute, and asked for whatever else
// its Python form has (__code__, __defaults__, ...).
struct Callable {
    PyObject_HEAD
    vectorcallfunc vectorcall;
    PyObject* slow;
    PyObject* dict;
    PyObject* weak;
    Op* op;
};

bool bound(const Op& op, Call& c, PyObject* const* args, Py_ssize_t n, PyObject* kwnames) {  // arguments to their places; false: not a call that the Python form would take either
    if (n > op.n) return false;
    for (Py_ssize_t i = 0; i < n; ++i) c.v[i] = args[i];
    const Py_ssize_t kw = kwnames ? PyTuple_GET_SIZE(kwnames) : 0;
    for (Py_ssize_t k = 0; k < kw; ++k) {
        PyObject* name = PyTuple_GET_ITEM(kwnames, k);
        int at = -1;
        for (int i = 0; i < op.n && at < 0; ++i)
            if (op.interned[i] == name) at = i;
        for (int i = 0; i < op.n && at < 0; ++i)
            if (PyUnicode_CompareWithASCIIString(name, op.args[i]) == 0) at = i;
        if (at < 0 || at < n) return false;
        c.v[at] = args[n + k];
    }
    return true;
}

PyObject* op_vectorcall(PyObject* self, PyObject* const* args, size_t nargsf, PyObject* kwnames) {
    Callable* f = reinterpret_cast<Callable*>(self);
    HANDLE_TH_ERRORS
    if (fn_device && at::impl::PythonTorchFunctionTLS::stack_len() == 0 && !c10::impl::TorchDispatchModeTLS::any_modes_set()) {
        Call c;
        c.home = PyFunction_Check(f->slow) ? PyFunction_GET_GLOBALS(f->slow) : nullptr;
        if (bound(*f->op, c, args, PyVectorcall_NARGS(nargsf), kwnames)) {
            try {
                return f->op->body(c);
            } catch (const Decline&) {
            } catch (const Raised&) {
                return nullptr;
            }
        }
    }
    if (dry) {  // (tests see what was left to Python)
        PyObject* left = Py_BuildValue("(ss)", "left", f->op->name);
        PyList_Append(dry, left);
        Py_DECREF(left);
    }
    return PyObject_Vectorcall(f->slow, args, nargsf, kwnames);
    END_HANDLE_TH_ERRORS
}
void op_dealloc(PyObject* self) {
    PyObject_GC_UnTrack(self);
    Callable* f = reinterpret_cast<Callable*>(self);
    if (f->weak) PyObject_ClearWeakRefs(self);
    Py_CLEAR(f->slow);
    Py_CLEAR(f->dict);
    PyObject_GC_Del(self);
}
int op_traverse(PyObject* self, visitproc visit, void* arg) {
    Callable* f = reinterpret_cast<Callable*>(self);
    Py_VISIT(f->slow);
    Py_VISIT(f->dict);
    return 0;
}
int op_clear(PyObject* self) {
    Callable* f = reinterpret_cast<Callable*>(self);
    Py_CLEAR(f->slow);
    Py_CLEAR(f->dict);
    return 0;
}
PyObject* op_repr(PyObject* self) { return PyUnicode_FromFormat("<native form of %R>", reinterpret_cast<Callable*>(self)->slow); }
PyObject* op_reduce(PyObject* self, PyObject*) { return PyObject_GetAttrString(self, "__qualname__"); }
PyObject* op_descr_get(PyObject* self, PyObject* of, PyObject*) { return of && of != Py_None ? PyMethod_New(self, of) : Py_NewRef(self); }
PyObject* op_getattro(PyObject* self, PyObject* name) {
    PyObject* own = PyObject_GenericGetAttr(self, name);
    if (own || !PyErr_ExceptionMatches(PyExc_AttributeError)) return own;
    PyErr_Clear();
    return PyObject_GetAttr(reinterpret_cast<Callable*>(self)->slow, name);
}
PyMethodDef op_methods[] = {{"__reduce__", op_reduce, METH_NOARGS, "by module and name, as a function"}, {}};
PyGetSetDef op_getset[] = {{"__dict__", PyObject_GenericGetDict, PyObject_GenericSetDict, nullptr, nullptr}, {}};
PyTypeObject op_type = {PyVarObject_HEAD_INIT(nullptr, 0)};

PyObject* operator_for(PyObject*, PyObject* args) {  // (name, Python form) -> the callable, or None
    const char* name;
    PyObject* slow;
    if (!PyArg_ParseTuple(args, "sO", &name, &slow)) return nullptr;
    for (int i = 0; i < n_ops; ++i)
        if (!strcmp(ops[i].name, name)) {
            Callable* f = PyObject_GC_New(Callable, &op_type);
            if (!f) return nullptr;
            f->vectorcall = op_vectorcall, f->slow = Py_NewRef(slow), f->dict = nullptr, f->weak = nullptr, f->op = &ops[i];
            PyObject_GC_Track(reinterpret_cast<PyObject*>(f));
            return reinterpret_cast<PyObject*>(f);
        }
    Py_RETURN_NONE;
}

PyObject* bind(PyObject*, PyObject* args) {
    const char* name;
    unsigned long long address;
    if (!PyArg_ParseTuple(args, "sK", &name, &address)) return nullptr;
    void* at = reinterpret_cast<void*>(address);
    if (!strcmp(name, "mi355_attn_bwd_workspace_bytes")) attn_bwd_workspace_bytes = reinterpret_cast<WorkspaceBytes>(at);
    if (!strcmp(name, "mi355_moe_choose_takes")) moe_choose_takes = reinterpret_cast<ChooseTakes>(at);
    if (!strcmp(name, "mi355_attn_bwd_split_bytes")) attn_bwd_split_bytes = reinterpret_cast<SplitBytes>(at);
    if (!strcmp(name, "mi355_attn_bwd_qnorm_partials")) attn_bwd_qnorm_partials = reinterpret_cast<Partials>(at);
    for (Slot* s : slots)
        if (!strcmp(s->name, name)) s->address = at;
    Py_RETURN_NONE;
}
PyObject* setup(PyObject*, PyObject* args) {  // (getDevice, getCurrentRawStream, set_device or None, fail)
    PyObject* f[4];
    if (!PyArg_ParseTuple(args, "OOOO", &f[0], &f[1], &f[2], &f[3])) return nullptr;
    PyObject** to[4] = {&fn_device, &fn_stream, &fn_set_device, &fn_fail};
    for (int i = 0; i < 4; ++i) Py_XSETREF(*to[i], f[i] == Py_None ? nullptr : Py_NewRef(f[i]));
    Py_RETURN_NONE;
}
PyObject* set_kernels(PyObject*, PyObject* o) {
    if (!PyDict_Check(o)) return PyErr_SetString(PyExc_TypeError, "a module's namespace"), nullptr;
    Py_XSETREF(kernels, Py_NewRef(o));
    Py_RETURN_NONE;
}
PyObject* set_dry(PyObject*, PyObject* o) {
    if (o != Py_None && !PyList_Check(o)) return PyErr_SetString(PyExc_TypeError, "a list, or None"), nullptr;
    Py_XSETREF(dry, o == Py_None ? nullptr : Py_NewRef(o));
    Py_RETURN_NONE;
}
PyObject* names(PyObject*, PyObject*) {
    PyObject* l = PyList_New(0);
    for (int i = 0; l && i < n_ops; ++i) {
        PyObject* s = Py_BuildValue("(si)", ops[i].name, ops[i].n);
        PyList_Append(l, s);
        Py_XDECREF(s);
    }
    return l;
}
PyObject* arguments(PyObject*, PyObject* o) {
    const char* name = PyUnicode_AsUTF8(o);
    if (!name) return nullptr;
    for (int i = 0; i < n_ops; ++i)
        if (!strcmp(ops[i].name, name)) {
            PyObject* l = PyList_New(ops[i].n);
            for (int k = 0; l && k < ops[i].n; ++k) PyList_SET_ITEM(l, k, PyUnicode_FromString(ops[i].args[k]));
            return l;
        }
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"operator_for", operator_for, METH_VARARGS, "operator_for(name, function): a callable that takes the function's calls natively where it can, or None"},
    {"bind", bind, METH_VARARGS, "bind(name, address): where an entry point of the loaded library is"},
    {"setup", setup, METH_VARARGS, "setup(getDevice, getCurrentRawStream, set_device, fail)"},
    {"set_kernels", set_kernels, METH_O, "set_kernels(namespace of kernels.py)"},
    {"dry", set_dry, METH_O, "dry(list): this thread's calls are appended to it as (entry point, arguments) instead of made, on tensors of any device; dry(None) ends that"},
    {"names", names, METH_NOARGS, "[(operator, number of arguments)]"},
    {"arguments", arguments, METH_O, "the names of an operator's arguments"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_wrap", "Native forms of the tensor-level launchers.", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__wrap() {
    op_type.tp_name = "llm_quest_amd._wrap.Operator";
    op_type.tp_basicsize = sizeof(Callable);
    op_type.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_GC | Py_TPFLAGS_HAVE_VECTORCALL;
    op_type.tp_vectorcall_offset = offsetof(Callable, vectorcall);
    op_type.tp_call = PyVectorcall_Call;
    op_type.tp_dealloc = op_dealloc;
    op_type.tp_traverse = op_traverse;
    op_type.tp_clear = op_clear;
    op_type.tp_repr = op_repr;
    op_type.tp_getset = op_getset;
    op_type.tp_dictoffset = offsetof(Callable, dict);
    op_type.tp_weaklistoffset = offsetof(Callable, weak);
    op_type.tp_methods = op_methods;
    op_type.tp_descr_get = op_descr_get;
    op_type.tp_getattro = op_getattro;
    op_type.tp_setattro = PyObject_GenericSetAttr;
    if (PyType_Ready(&op_type) < 0) return nullptr;
    for (int i = 0; i < n_ops; ++i)
        for (int k = 0; k < ops[i].n; ++k)
            if (!(ops[i].interned[k] = PyUnicode_InternFromString(ops[i].args[k]))) return nullptr;
    PyObject* m = PyModule_Create(&module);
    if (m && PyModule_AddStringConstant(m, "torch_version", TORCH_VERSION) < 0) return nullptr;
    return m;
}
