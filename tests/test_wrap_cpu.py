"""The native forms of the launchers (csrc/wrap.cpp) against their Python forms, without a GPU: what each would hand to the library, and what it returns, over the forms that a call may have -- strides,
optional operands, types, odd sizes -- and over calls that the Python form refuses, which the native one must leave to it."""
import copy
import functools
import inspect
import itertools
import pickle
import weakref

import pytest
import torch

from llm_quest_amd import _lib as L
from llm_quest_amd import kernels as K
from llm_quest_amd import kernels_q35 as Q
from llm_quest_amd import kernels_seq as S
from llm_quest_amd import ops_decode as O

if L._wrap is None:
    pytest.skip("the extension is not built", allow_module_level=True)
B, F, I, U, I64 = torch.bfloat16, torch.float32, torch.int32, torch.uint8, torch.int64


def form(name):
    for m in (K, Q, S, O):
        f = getattr(m, name, None)
        if f is not None and hasattr(f, "__wrapped__") and f.__wrapped__.__module__ == m.__name__:
            return f
    raise KeyError(name)


@pytest.fixture
def both(monkeypatch):
    """check(name, *args, **kw): the two forms' calls and results are alike; returns whether the native one took the call."""
    L.load()
    made = {}

    def scratch(device, nbytes=64):
        return made.setdefault(nbytes, torch.empty(nbytes, dtype=U))

    monkeypatch.setattr(K, "_workspace", lambda device: made.setdefault("ws", torch.empty(64)))
    monkeypatch.setattr(K, "_attn_scratch", scratch)
    monkeypatch.setattr(K, "rope_cs16", lambda cos, sin: made.setdefault("cs", torch.zeros(4, dtype=B)))
    known = set()  # addresses that the call came with: the others are outputs', told by their order

    def told(calls):
        seen, out = {}, []
        for name, *args in calls:
            row = [name]
            for a in args:
                if isinstance(a, int) and a > 1 << 20 and a not in known and a != K.WS_BYTES:
                    a = seen.setdefault(a, f"output {len(seen)}")
                row.append(a)
            out.append(row)
        return out

    def facts(r):
        if isinstance(r, (tuple, list)):
            return [facts(x) for x in r]
        if torch.is_tensor(r):
            return (tuple(r.shape), r.stride(), r.dtype, r.data_ptr() if r.data_ptr() in known else None)
        return r

    def check(name, *args, **kw):
        f = form(name)
        known.clear()

        def note(x):
            if torch.is_tensor(x):
                known.add(x.data_ptr())
            elif isinstance(x, (tuple, list)):
                for y in x:
                    note(y)

        note(args), note(list(kw.values())), note(list(made.values()))
        native, slow = [], []
        L._wrap.dry(native)
        try:
            with monkeypatch.context() as m:
                m.setattr(L, "call", lambda n, *a: native.append(("python",)) or None)
                m.setattr(L, "require_gpu", lambda *t: None)
                try:
                    got = f(*args, **kw)
                except Exception as e:
                    got = e
        finally:
            L._wrap.dry(None)
        note(list(made.values()))
        with monkeypatch.context() as m:
            m.setattr(L, "call", lambda n, *a: slow.append((n, *(int(x) if isinstance(x, bool) else x for x in a))))
            m.setattr(L, "require_gpu", lambda *t: None)
            for op, _ in L._wrap.names():  # a Python form calls Python forms
                g = form(op)
                m.setattr(inspect.getmodule(g.__wrapped__), op, g.__wrapped__)
            try:
                want = f.__wrapped__(*args, **kw)
            except Exception as e:
                want = e
        if native and native[0] == ("left", name):
            assert type(got) is type(want), (name, got, want)
            return False
        assert not isinstance(want, Exception), (name, "taken where Python says", want)
        problems = [list(c) for c in slow]
        if name == "gemm_grouped":  # the table's address is its own; its entries are read
            assert [c[:3] + [c[4]] for c in told(native)] == [[c[0], c[1], c[2], c[4]] for c in problems]
        else:
            a, b = told(native), told(problems)
            assert len(a) == len(b), (name, a, b)
            for x, y in zip(a, b):
                assert x[0] == y[0] and len(x) == len(y), (x, y)
                for i, (u, v) in enumerate(zip(x[1:], y[1:])):
                    assert u == v or (v is None and u in (None, 0)) or (isinstance(v, float) and torch.tensor(u, dtype=F) == torch.tensor(v, dtype=F)), (name, i, u, v, x, y)
        assert facts(got) == facts(want), (name, facts(got), facts(want))
        return True

    return check


def rows(r, c, dtype=B, pad=0):
    return torch.randn(r, c + pad).to(dtype)[:, :c]


def ints(n):
    return torch.arange(n, dtype=I)


def test_operators_are_what_functions_are_besides_being_called():
    class Holder:
        product = K.gemm

    for name, _ in L._wrap.names():
        f, slow = form(name), form(name).__wrapped__
        assert pickle.loads(pickle.dumps(f)) is f and copy.deepcopy(f) is f and copy.copy(f) is f and weakref.ref(f)() is f
        assert f.__name__ == name and f.__code__ is slow.__code__ and f.__defaults__ == slow.__defaults__ and f.__globals__ is slow.__globals__ and inspect.signature(f) == inspect.signature(slow)
        assert not hasattr(f, "nothing") and f.__doc__ == slow.__doc__
    module = torch.nn.Module()
    module.product, module.half = K.gemm, functools.partial(K.gemm, L.GEMM_NT)
    copied = copy.deepcopy(module)
    assert copied.product is K.gemm and copied.half.func is K.gemm and copied.half.args == (L.GEMM_NT,) and pickle.loads(pickle.dumps(copied.half)).func is K.gemm
    h = Holder()
    assert Holder.product is K.gemm and inspect.ismethod(h.product) and h.product.__self__ is h and h.product.__func__ is K.gemm


def test_a_dry_run_is_one_threads_own():
    import threading

    calls, seen = [], []

    def other():
        try:
            K.gelu_fwd(torch.randn(8).to(B))
        except Exception as e:  # (no GPU tensor)
            seen.append(type(e))

    L._wrap.dry(calls)
    try:
        t = threading.Thread(target=other)
        t.start()
        t.join()
        K.copy2d(rows(2, 8), rows(2, 8))
    finally:
        L._wrap.dry(None)
    assert seen and [c[0] for c in calls] == ["mi355_copy2d"]


def test_arguments_are_named_as_in_python():
    for name, _ in L._wrap.names():
        assert list(inspect.signature(form(name)).parameters) == L._wrap.arguments(name), name


@pytest.mark.parametrize("M,N,Kd", [(1, 8, 8), (9, 40, 24), (130, 64, 256)])
def test_products(both, M, N, Kd):
    shapes = {L.GEMM_NT: ((M, Kd), (N, Kd)), L.GEMM_NN: ((M, Kd), (Kd, N)), L.GEMM_TN: ((Kd, M), (Kd, N))}
    for form_, pad, odt in itertools.product(shapes, (0, 8), (B, F)):
        a, b = (rows(*s, pad=pad) for s in shapes[form_])
        assert both("gemm", form_, a, b, out_dtype=odt)
        assert both("gemm", form_, a, b, None, odt, torch.randn(N), rows(M, N, odt, pad), True, False)
        assert both("gemm", form_, a, b, out=rows(M, N, odt, 3), residual=rows(M, N, odt))
    a, b = rows(M, Kd), rows(N, Kd)
    for bad in (dict(bias=torch.randn(N + 1)), dict(bias=torch.randn(N).to(B)), dict(bias=torch.randn(2 * N)[::2]), dict(residual=rows(M, N, F)), dict(residual=rows(M + 1, N)), dict(out=rows(M, N + 1)), dict(out=rows(N, M).t()),
                dict(tile=1), dict(split3_out=True), dict(out_dtype=None), dict(out_dtype=torch.float16)):
        assert not both("gemm", L.GEMM_NT, a, b, **bad) or (M == 1 and "out" in bad and bad["out"].shape == (M, N))
    assert not both("gemm", L.GEMM_NT, a.float(), b) and not both("gemm", L.GEMM_NT, a, rows(N, Kd + 8)) and not both("gemm", L.GEMM_NT, a[0], b) and not both("gemm", 3, a, b)
    assert not both("gemm", L.GEMM_NT, rows(Kd, M).t() if M > 1 else a[0], b)
    assert both("dgrad", rows(M, N), rows(N, Kd)) and both("dgrad", rows(M, N), rows(N, Kd, pad=8), rows(M, Kd)) and not both("dgrad", rows(M, N), rows(N + 1, Kd))
    dy, x = rows(Kd, M), rows(Kd, N)
    for odt in (B, F):
        assert both("gemm_grouped", L.GEMM_TN, [(dy, x, rows(M, N, odt), None), (dy, x, rows(M, N, odt), rows(M, N, odt))])
    assert not both("gemm_grouped", L.GEMM_TN, [(dy, x, rows(M, N), None), (dy, x, rows(M, N, F), None)])
    assert not both("gemm_grouped", L.GEMM_TN, [(dy, x, rows(M, N), None)] * 9) and not both("gemm_grouped", L.GEMM_TN, [])


def test_products_that_the_persistent_kernel_may_take_are_counted_in_python(both, monkeypatch):
    a, b = torch.empty(4096, 128, dtype=B), torch.empty(8192, 128, dtype=B)  # 16 x 32 tiles
    assert not both("gemm", L.GEMM_NT, a, b) and both("gemm", L.GEMM_NT, a[:3840], b) and both("gemm", L.GEMM_NT, a[:, :64], b[:, :64]) and both("gemm", L.GEMM_NT, a, b, bias=torch.zeros(8192))
    assert not both("gemm_gateup_swiglu", a, b) and both("gemm_gateup_swiglu", a[:256], b)
    monkeypatch.setattr(K, "_PERSIST_USER", "1")
    assert not both("gemm", L.GEMM_NT, a[:256], b)
    monkeypatch.setattr(K, "_PERSIST_USER", None)
    for knob in ("_TILE_OVERRIDE", "_TILE_NT_PLAIN"):
        with monkeypatch.context() as m:
            m.setattr(K, knob, 1)
            assert not both("gemm", L.GEMM_NT, a[:256], b)
    monkeypatch.setattr(K, "_TILE_BY_FORM", {0: 0, 1: 0, 2: 5})
    assert not both("gemm", L.GEMM_TN, a, a) and both("gemm", L.GEMM_NT, a[:256], b)


def test_constants_are_read_where_the_python_form_reads_them(both, monkeypatch):
    """One that is changed in its module holds for both forms: the same calls, or none natively."""
    monkeypatch.setattr(K, "transpose", lambda w: w.t().contiguous())
    dy, w = rows(600, 64), rows(64, 40)
    assert both("dgrad", dy, w) and both("dgrad", torch.empty(1279, 4096, dtype=B), torch.empty(4096, 1024, dtype=B))  # (a row more is transposed)
    with monkeypatch.context() as m:
        m.setattr(K, "DGRAD_NT_MIN_ROWS", 512)
        assert not both("dgrad", dy, w) and both("dgrad", dy[:511], w)
        m.setattr(K, "DGRAD_NT_MIN_ROWS", 1 << 20)
        assert not both("dgrad", rows(1280, 64), w) and both("dgrad", rows(1279, 64), w)
    x, g = rows(40, 16), rows(40, 16)
    for parts in (3, 512):
        monkeypatch.setattr(K, "NORM_PARTS", parts)
        monkeypatch.setattr(K, "QK_PARTS", parts)
        monkeypatch.setattr(Q, "NORM_PARTS", 8 * parts)
        monkeypatch.setattr(Q, "CONV_TOKEN_CHUNK", parts + 4)
        assert both("rmsnorm_bwd", x, torch.randn(16).to(B), torch.randn(40), g)
        assert both("gated_rmsnorm_bwd", x, torch.randn(8), x, torch.randn(40, 2), g, rows(40, 16), 2, 8)
        assert both("headnorm_rope_bwd", x, 2, 8, 8, torch.randn(8).to(B), None, None, None, torch.randn(40, 2), g, rows(40, 16), 8)
        assert both("qknorm_rope_bwd", rows(40, 6 * 64), None, None, None, None, None, None, None, rows(40, 64), rows(40, 6 * 64), 4, 1, 64)
        assert both("causal_conv_silu_bwd", x, torch.randn(16, 1, 4).to(B), g, rows(40, 16), 2, 20)
    monkeypatch.setattr(Q, "CONV_TOKEN_CHUNK", "thirty")
    assert not both("causal_conv_silu_bwd", x, torch.randn(16, 1, 4).to(B), g, rows(40, 16), 2, 20)


def test_training_rows(both):
    for M, W in ((1, 8), (37, 256)):
        x, w, g = rows(M, W), torch.randn(W).to(B), rows(M, W)
        assert both("rmsnorm_fwd", x, w) and both("rmsnorm_fwd", x, w, 1e-5, want_rstd=False) and not both("rmsnorm_fwd", rows(M, W, pad=8) if M > 1 else x.float(), w) and not both("rmsnorm_fwd", x, w[:-1])
        r = torch.randn(M)
        assert both("rmsnorm_bwd", x, w, r, g) and both("rmsnorm_bwd", x, w, r, g, dres=g, dw_out=torch.zeros(W), dw_accumulate=True) and both("rmsnorm_bwd", x, w, r, g, dw_out=torch.zeros(W, dtype=B))
        assert both("rmsnorm_bwd", x, w, r, g, dres=g, partial=True)
        assert not both("rmsnorm_bwd", x, w, r, g.float()) and not both("rmsnorm_bwd", x, w, r, rows(M + 1, W)) and not both("rmsnorm_bwd", x, w, r, g, dres=rows(M, W, F))
        assert both("swiglu_fwd", rows(M, 2 * W), W) and both("swiglu_bwd", rows(M, 2 * W), g, W) and not both("swiglu_fwd", x, W) and not both("swiglu_bwd", rows(M, 2 * W), rows(M, W + 1), W)
        xf, s = rows(M, W, F), torch.randn(W)
        for dt, st in itertools.product((B, F), (False, True)):
            assert both("layernorm_fwd", xf, s, s, out_dtype=dt, want_stats=st)
        assert not both("layernorm_fwd", xf, s, s, out_dtype="split3") and not both("layernorm_fwd", x, s, s) and not both("layernorm_fwd", xf, s, w) and not both("layernorm_fwd", xf, s, s, None)
        d = [(torch.zeros(W), True), None, (torch.zeros(W), False)]
        for dy in (g, xf):
            assert both("layernorm_bwd_bf16", xf, s, r, r, dy, xf, d) and both("layernorm_bwd_bf16", xf, s, r, r, dy, None, tuple(d), eps=1e-6, mode=1)
        one = torch.zeros(W)
        assert not both("layernorm_bwd_bf16", xf, s, r, r, g, xf, [(one, True), None, (one, True)]) and not both("layernorm_bwd_bf16", xf, s, r, r, g, xf, [(w, True), None, None])
        sums = [(rows(5, W, F), torch.zeros(W, dtype=B), True), (rows(1, W, F, 8), torch.zeros(W), False), (rows(7, 2 * W, F)[:, W:], torch.zeros(W, dtype=B), False), (rows(2, 8, F), torch.zeros(2, 4), True)]
        assert all(both("reduce_rows_each", sums[:n]) for n in (1, 2, 3, 4)) and not both("reduce_rows_each", []) and not both("reduce_rows_each", sums + sums[:1])
        assert not both("reduce_rows_each", [(rows(5, W, F), torch.zeros(W + 1), True)]) and not both("reduce_rows_each", [(rows(5, W), torch.zeros(W), True)])
        assert both("reduce_rows_into", rows(3, 2 * W, F), 3, W, [(one, False), (torch.zeros(W), True)]) and not both("reduce_rows_into", rows(3, W, F), 3, W, [None])
        assert both("gelu_fwd", x) and both("gelu_fwd", x, tanh=True) and not both("gelu_fwd", xf) and both("gelu_bwd_colsum", x, g, (one, True)) and not both("gelu_bwd_colsum", x, g, None)
        assert both("colsum", rows(M, W, pad=4)) and both("colsum", xf, one, True) and not both("colsum", x, torch.zeros(W + 1)) and both("add_f32_to_bf16", one, None, w) and both("add_f32_to_bf16", one, w, w)
        assert both("copy2d", rows(M, W, pad=8), x) and both("copy2d", xf, rows(M, W, F, 4)) and not both("copy2d", x, xf) and not both("copy2d", x, rows(M, W + 1))
        if W % 64 == 0:
            assert both("gemm_gateup_swiglu", x, rows(128, W)) and not both("gemm_gateup_swiglu", x, rows(96, W)) and both("gemm_dgrad_swiglu_bwd", rows(M, 40), rows(40, W), rows(M, 2 * W))
            assert not both("gemm_dgrad_swiglu_bwd", rows(M, 40), rows(40, W), rows(M, 2 * W, pad=8)) or M == 1


@pytest.mark.parametrize("D", [64, 128])
def test_attention(both, D, monkeypatch):
    Bn, Sn, Hq, Hkv = 2, 5, 4, 2
    T = Bn * Sn
    qkv, cs, pos = rows(T, (Hq + 2 * Hkv) * D), torch.randn(9, D), ints(T)
    qw, kw = torch.randn(D).to(B), torch.randn(D).to(B)
    assert both("qknorm_rope_fwd", qkv, qw, kw, cs, cs, pos, Hq, Hkv, D) and both("qknorm_rope_fwd", qkv, None, None, cs, cs, pos, Hq, Hkv, D, eps=1e-5)
    assert not both("qknorm_rope_fwd", qkv, qw, kw, cs, cs, pos.long(), Hq, Hkv, D) and not both("qknorm_rope_fwd", qkv, qw, kw, cs[:, :-1], cs, pos, Hq, Hkv, D)
    q, k, v, o, do = rows(T, Hq * D), rows(T, Hkv * D), qkv[:, (Hq + Hkv) * D :], rows(T, Hq * D), rows(T, Hq * D)
    lse, mask, rstd = torch.randn(Bn, Hq, Sn), torch.ones(Bn, Sn, dtype=U), torch.randn(T, Hq + Hkv)
    for name in ("attn_fwd", "attn_generic_fwd"):
        assert both(name, q, k, v, Bn, Sn, Hq, Hkv, D) and both(name, q, k, v, Bn, Sn, Hq, Hkv, D, key_mask=mask, scale=0.3) and not both(name, q, k, v, Bn, Sn, Hq, Hkv, D, key_mask=mask.bool())
        assert not both(name, q.float(), k, v, Bn, Sn, Hq, Hkv, D) and not both(name, q, k, v, Bn, Sn + 1, Hq, Hkv, D)
    assert both("attn_fwd", q, k, v, Bn, Sn, Hq, Hkv, D, None, False, None)
    dq, dk, dqkv = rows(T, Hq * D), rows(T, Hkv * D), rows(T, (Hq + 2 * Hkv) * D)
    dv = dqkv[:, (Hq + Hkv) * D :]
    for name in ("attn_bwd", "attn_generic_bwd"):
        assert both(name, q, k, v, o, do, lse, Bn, Sn, Hq, Hkv, D, dq, dk, dv) and both(name, q, k, v, o, do, lse, Bn, Sn, Hq, Hkv, D, dq, dk, dv, key_mask=mask, scale=0.1)
        assert not both(name, q, k, v, o, do, lse[:1], Bn, Sn, Hq, Hkv, D, dq, dk, dv)
    monkeypatch.setattr(K, "_ATTN_DS_SPILL", False)
    assert both("attn_bwd", q, k, v, o, do, lse, Bn, Sn, Hq, Hkv, D, dq, dk, dv, None, False)
    monkeypatch.setattr(K, "_ATTN_DS_SPILL", True)
    for a in (dq, None):
        assert both("qknorm_rope_bwd", qkv, qw, kw, cs, cs, pos, rstd, a, dk, dqkv, Hq, Hkv, D) and both("qknorm_rope_bwd", qkv, qw, kw, cs, cs, pos, rstd, a, dk, dqkv, Hq, Hkv, D, True)
    args = (q, k, v, o, do, lse, Bn, Sn, Hq, Hkv, D, dk, dv, qkv, qw, cs, cs, pos, rstd, dqkv)
    taken = D == 128
    assert both("attn_bwd_qnorm", *args) is taken and both("attn_bwd_qnorm", *args, partial=True) is taken and both("attn_bwd_qnorm", *args, key_mask=mask, causal=True, scale=0.2, delta=torch.randn(Bn, Hq, Sn)) is taken
    assert not both("attn_bwd_qnorm", *args[:14], None, *args[15:]) and not both("attn_bwd_qnorm", *args, delta=lse[:, :1])
    monkeypatch.setattr(K, "_attn_scratch", lambda d, n: None)
    assert not both("attn_bwd_qnorm", *args) and both("attn_bwd", q, k, v, o, do, lse, Bn, Sn, Hq, Hkv, D, dq, dk, dv)


def test_hybrid_rows(both):
    T, H, D = 6, 3, 16
    assert both("zc_weight", torch.randn(9).to(B)) and not both("zc_weight", torch.randn(9))
    wide, cs, pos, w = rows(T, 2 * H * D + 5), torch.randn(T, 8), ints(T), torch.randn(D).to(B)
    assert both("headnorm_rope_fwd", wide, H, D, 2 * D, w, cs, cs, pos) and both("headnorm_rope_fwd", wide, H, D, D, w, None, None, None) and not both("headnorm_rope_fwd", wide, H, D, 3 * D, w, cs, cs, pos)
    rstd, dout = torch.randn(T, H), rows(T, H * D)
    assert both("headnorm_rope_bwd", wide, H, D, 2 * D, w, cs, cs, pos, rstd, dout, rows(T, H * D), D) and both("headnorm_rope_bwd", wide, H, D, 2 * D, w, cs, cs, pos, rstd, dout, rows(T, H * D), D, True) and not both("headnorm_rope_bwd", wide, H, D, 2 * D, w, cs, cs, pos, rstd, dout.float(), rows(T, H * D), D)
    ctx = rows(T, H * D)
    assert both("sigmoid_gate_fwd", ctx, wide, H, D, 2 * D) and both("sigmoid_gate_bwd", ctx, wide, H, D, 2 * D, dout, rows(T, 2 * H * D), 2 * D) and not both("sigmoid_gate_fwd", ctx, wide.float(), H, D, D)
    both_ = rows(T, 2 * H)
    b, a, A, dt = both_[:, :H], both_[:, H:], torch.randn(H), torch.randn(H).to(B)
    g = torch.randn(T, H)
    assert both("gdn_gates_fwd", b, a, A, dt) and not both("gdn_gates_fwd", b, rows(T, H), A, dt) and both("gdn_gates_bwd", b, a, A, dt, g, g, both_[:, :H], both_[:, H:])
    assert both("gdn_gates_bwd", b, a, A, dt, g, g, both_[:, :H], both_[:, H:], partial=True)
    assert not both("gdn_gates_bwd", b, a, A, dt, g, g.to(B), both_[:, :H], both_[:, H:])
    x, cw = wide[:, : H * D], torch.randn(H * D, 1, 4).to(B)
    assert both("causal_conv_silu_fwd", x, cw, 2, 3) and not both("causal_conv_silu_fwd", x, cw, 2, 4) and not both("causal_conv_silu_fwd", x, cw.float(), 2, 3)
    assert both("causal_conv_silu_bwd", x, cw, dout, rows(T, H * D), 2, 3, True)
    assert both("causal_conv_silu_bwd", x, cw, dout, rows(T, H * D), 2, 3) and both("causal_conv_silu_bwd", x, cw, dout, x, 2, 3) and both("causal_conv_silu_bwd", x, cw, dout, dout, 2, 3)
    assert both("l2norm_fwd", x, H, D) and both("l2norm_bwd", x, dout, x, H, D) and not both("l2norm_fwd", x, H, D + 1) and not both("l2norm_bwd", x, dout.float(), x, H, D)
    wf = torch.randn(D)
    assert both("gated_rmsnorm_bwd", ctx, wf, x, rstd, dout, rows(T, H * D), H, D, True)
    assert both("gated_rmsnorm_fwd", ctx, wf, x, H, D) and both("gated_rmsnorm_bwd", ctx, wf, x, rstd, dout, rows(T, H * D), H, D) and not both("gated_rmsnorm_fwd", ctx, w, x, H, D)


@pytest.mark.parametrize("M", [1, 8, 9])
@pytest.mark.parametrize("dtype", [B, F])
def test_linear(both, M, dtype):
    for Kd, pad in ((16, 0), (16, 8), (16, 4), (12, 0)):
        x, w = rows(M, Kd, dtype, pad), rows(24, Kd, B, pad)
        for od, bias in itertools.product((None, B, F), (None, torch.randn(24))):
            assert both("linear", x, w, od, bias)
    x, w = rows(M, 16, dtype), rows(24, 16)
    assert both("linear", x[:, :8], w[:, 8:], out_dtype=F)
    assert not both("linear", x, w.float()) and not both("linear", x, rows(24, 8)) and not both("linear", x, w, torch.float16) and not both("linear", x, w, F, torch.randn(24).to(B))
    if dtype == B:
        assert both("gemv", x, w) is (M <= 8) and both("gemv", x, w, rows(M, 24)) is (M <= 8) and not both("gemv", x.float(), w)


def test_served_rows(both):
    T, W, n = 5, 16, 4
    x3, x2, v, m, r = torch.randn(T, n, W), torch.randn(T, W), torch.randn(n), torch.randn(n, n), torch.tensor([0, 3])
    nw = torch.randn(W)
    for x in (x3, x2):
        assert both("hyper_mix", x, n, read=v, norm=nw, eps=1e-6, out_dtype=B, x_out=None) and both("hyper_mix", x, n, read=v, want_u=True)
        for y in (rows(2 * T, W), rows(2 * T, W, F, 4)):
            assert both("hyper_mix", x, n, y=y, parts=2, y_scale=0.5, mix=m, put=v, read=v, norm=nw, eps=1e-5, x_out=True) and both("hyper_mix", x, n, y, 2, mix=m, put=v, x_out=torch.empty(T, n, W))
        assert both("hyper_mix", x, n, read=v, rows=r, norm=nw) and not both("hyper_mix", x, n, read=v, rows=r.int()) and not both("hyper_mix", x, n, y=rows(T, W)) and not both("hyper_mix", x, n, read=nw)
        assert not both("hyper_mix", x.to(B), n, read=v) and not both("hyper_mix", x, n, read=v, norm=nw, out_dtype=torch.float16) and not both("hyper_mix", x, n, read=v, x_out=torch.empty(T, n, W + 1))
    for na, nb in itertools.product((None, (nw, B, False), (nw, None, True), (nw, F, True), (nw, B, True)), (None, (nw, F, False))):
        assert both("group_rmsnorm_sum", x2, 2, 1e-6, norm_a=na, norm_b=nb) and both("group_rmsnorm_sum", x2, 2, 1e-6, y1=rows(T, W), y2=rows(3 * T, W, F, 2), parts=3, x_out=True, norm_a=na, norm_b=nb)
    got = S.group_rmsnorm_sum
    assert both("group_rmsnorm_sum", x2, 1, 1e-6, y1=x2, x_out=x2) and not both("group_rmsnorm_sum", x2, 1, 1e-6, y1=rows(T, W + 1)) and not both("group_rmsnorm_sum", x2, 1, 1e-6, norm_a=(nw[1:], B, False)) and got
    off, slot, rs = torch.tensor([0, 2, 5], dtype=I), ints(2), torch.tensor([0, 0, 1, 1, 1], dtype=I)
    for dt, od, bias in itertools.product((B, F), (None, B, F), (None, nw)):
        assert both("ragged_conv", rows(T, W, dt, 4), torch.randn(W, 4), torch.zeros(2, 3, W), rs, off, slot, act=True, residual=True, out_dtype=od, bias=bias)
    assert both("ragged_conv", x2, torch.randn(W, 1), None, rs, off, slot) and not both("ragged_conv", x2, torch.randn(W, 4), torch.zeros(2, 2, W), rs, off, slot) and not both("ragged_conv", x2, torch.randn(W, 4), None, rs, off, slot)
    assert both("gated_headnorm", x2, nw[:8], rows(T, W, B, 3), 2, 8, 1e-6, B) and both("gated_headnorm", x2, nw[:8], x2, 2, 8, 1e-6, F) and not both("gated_headnorm", x2, nw, x2, 2, 8, 1e-6, B)
    for dt in (B, F):
        assert both("glu_rows", rows(T, W, dt, 2), S.GLU_SILU) and both("glu_rows", rows(T, W, dt), S.GLU_CLAMPED_SWISH, 7.0, F) and both("rmsnorm_rows", rows(T, W, dt, 4), nw, 1e-6) and both("rmsnorm_rows", x2, nw, 1e-6, dt)
        for cast in (None, B, F):
            assert both("add_layernorm", x2, nw, nw, 1e-6, 0.5, rows(2 * T, W, dt, 4), 2, cast) and both("add_layernorm", x2, nw, nw, 1e-6, cast_dtype=cast)
    assert not both("add_layernorm", x2, nw, nw[1:], 1e-6) and not both("rmsnorm_rows", x2, nw[1:], 1e-6)
    assert both("unary_rows", x2, S.UNARY_SOFTCAP, limit=30.0) and both("unary_rows", x2, S.UNARY_TANH, out_dtype=B) and not both("unary_rows", x2, S.UNARY_HEAD_GATE, gate=rows(T, 2), group=8)
    tab = torch.randn(9, W).to(B)
    assert both("embed_hash", ints(T), ints(T), tab, 2.0) and both("embed_hash", ints(T), ints(T), tab, 1.0, torch.randn(8, W).to(B), 7, 31, 7) and both("embed_hash", ints(T), None, tab, 1, out=torch.empty(T, W))
    assert not both("embed_hash", ints(T).long(), None, tab, 1.0) and not both("embed_hash", ints(T), ints(T), tab, 1.0, torch.randn(8, W).to(B), 9)
    lg = torch.randn(T, 8)
    assert both("router_logits", x2, rows(8, W)) and both("moe_route", lg, None, 2, 1, 1, 1.0, softmax=True) and both("moe_route", lg, torch.randn(8), 2, 4, 2, 2.5) and not both("moe_route", lg, torch.randn(8), 2, 1, 1, 1.0, softmax="chosen")
    for n, corr in itertools.product((3, 8, 9), (None, torch.randn(8))):  # (from nine tokens on three launches)
        assert both("moe_choose", torch.randn(n, W), rows(8, W), corr, 2, 4, 2, 2.5) and both("moe_choose", torch.randn(n, W), rows(8, W), corr, 2, 1, 1, 1.0, True)
    assert not both("moe_choose", x2, rows(8, W), None, 2, 1, 1, 1.0, "chosen") and not both("moe_choose", x2, rows(8, W + 8), None, 2, 1, 1, 1.0)
    assert both("moe_dispatch", ints(10), 8) and not both("moe_dispatch", ints(10).long(), 8)
    out = torch.empty(T, 24)
    assert both("bgemm", x2, rows(24, W), out, T, 24, W) and both("bgemm", rows(T, W), rows(24, W), out, T, 24, W, batch=2, lda=W, a_bs=1, sbn=W, sbk=1, b_bs=3, ldc=24, c_bs=2, mfma=False, bias=torch.randn(24), limit=3, n_out=12)
    assert both("bgemm", rows(T, W), rows(24, W), out, T, 24, W, grp_offs=off, a_rows=rs, a_div=2, c_rows=rs, row_scale=nw, epi=4) and not both("bgemm", x2, rows(24, W), out, T, 24, W, bias=torch.randn(23))


def test_served_attention(both):
    T, H, G, d, dv = 5, 4, 2, 16, 16
    pos, dst, cache = ints(T), ints(T), torch.zeros(64, G * (d + dv), dtype=B)
    wide = rows(T, (H + 2 * G) * d + 7, F)
    src = wide[:, : (H + 2 * G) * d]
    vecs = dict(qw=torch.randn(d), kw=torch.randn(d), qscale=torch.randn(H), freq=torch.randn(d // 2))
    for dt in (B, F):
        c = cache.to(dt)
        assert both("qkv_rows_append", src, H, G, d, dv, None, vecs["qw"], vecs["kw"], 1e-6, vecs["qscale"], d, 1, vecs["freq"], pos, dst, c)
        assert both("qkv_rows_append", src, H, G, d, dv, torch.randn((H + 2 * G) * d), None, None, 1e-6, None, 0, 0, None, pos, dst, c, vmix=rows(T, G * dv, F, 3), lam=0.3, unit_norm=True, rot_amp=1.1)
        assert both("qkv_rows_append", src[:, : (H + G) * d], H, G, d, dv, None, None, None, 1e-6, None, d, 0, vecs["freq"], pos, dst, c, tie_v=True)
    assert not both("qkv_rows_append", src, H, G, d, dv, None, None, None, 1e-6, None, 0, 0, None, pos, dst, cache, q_temp=(0.1, 4)) and not both("qkv_rows_append", src[:, 1:], H, G, d, dv, None, None, None, 1e-6, None, 0, 0, None, pos, dst, cache)
    assert not both("qkv_rows_append", src, H, G, d, dv, None, None, None, 1e-6, None, d, 0, vecs["freq"][1:], pos, dst, cache)
    q, one = torch.randn(T, H * d), ints(2)
    desc = (one, one, one, one, one, one)
    for dt, odt in ((B, B), (B, F), (F, F)):
        c, out = cache.to(dt), torch.empty(T, H * dv, dtype=odt)
        for max_new, max_keys, window, keep, chunk in itertools.product((1, 3, 200), (0, 40, 700, 9000), (0, 512), (0, 4), (0, 128)):
            assert both("latent_attn", q, c, None, c[:, G * d :], out, H, 2, d, 0, dv, d, d, dv, dv, desc, max_new, 0.25, max_keys=max_keys, kv_rep=H // G, window=window, keep_first=keep, softcap=50.0, chunk=chunk)
        assert both("latent_attn", q, c, c[:, :4], c[:, G * d :], out, H, 2, d, 4, dv, d, d, dv, dv, desc, 1, 0.25, 5000, sink=torch.randn(H), sig_bias=torch.randn(H), slope=torch.randn(H), gate=rows(T, H * dv, F, 5))
    out = torch.empty(T, H * dv, dtype=B)
    assert not both("latent_attn", q, cache, None, cache, out, H, 2, d, 0, dv, d, d, dv, dv, desc, 1, 0.25, pool=4, pooled=(cache, cache), pool_row0=one) and not both("latent_attn", q, cache, None, cache, out, H, 2, d, 0, dv, d, d, dv, dv, desc, 1, 0.25, slope=torch.randn(H + 1))
    assert not both("latent_attn", q.to(B), cache, None, cache, out, H, 2, d, 0, dv, d, d, dv, dv, desc, 1, 0.25) and not both("latent_attn", q, cache, None, cache, out, H, 2, d, 0, dv, d, d, dv, dv, desc[:5] + (one.long(),), 1, 0.25)
    lat, lc = rows(T, 12, F, 4), torch.zeros(64, 12, dtype=B)
    assert both("latent_kv_append", lat, 8, 4, torch.randn(8), 1e-6, pos, dst, torch.randn(2), 4, lc) and both("latent_kv_append", lat, 8, 4, torch.randn(8), 1e-6, pos, dst, None, 0, lc, layout=1)
    assert not both("latent_kv_append", lat, 8, 4, torch.randn(8), 1e-6, pos, dst, torch.randn(1), 4, lc)
    o = torch.empty(T, H * d)
    assert both("rope_heads", wide, H, d, d, 2, o, d, 0, 0, 8, vecs["freq"], pos) and both("rope_heads", rows(T, H * d), H, d, d, 0, o, d, 0, 0, 8, vecs["freq"], pos, layout=1) and not both("rope_heads", o, H, d, d, 2, o, d, 0, 0, 8, vecs["freq"], pos)
    st, off = torch.zeros(2, H, d, dv), torch.tensor([0, 2, 5], dtype=I)
    for dt, zt in itertools.product((B, F), (B, F)):
        q2, z = rows(T, H * d, dt, 4), rows(T, H * d, zt)
        assert both("gla", q2, q2, rows(T, H * dv, dt), z, torch.randn(H * d), 1 / 16.0, 0.25, off, one, st, H, d, dv)
    assert not both("gla", q, q, q, None, None, 1.0, 0.25, off, one, st, H, d, dv, head_decay=torch.rand(H)) and not both("gla", q, q, q, q, torch.randn(H * d), 1.0, 0.25, off, one, st[:, :, 1:], H, d, dv)


def test_other_tensors_and_modes_go_to_python(both):
    class Mine(torch.Tensor):
        pass

    x, w = rows(4, 16), torch.randn(16).to(B)
    assert not both("rmsnorm_fwd", x.as_subclass(Mine), w) and both("rmsnorm_fwd", x, torch.nn.Parameter(w)) and not both("rmsnorm_fwd", x, w, "1e-6") and not both("rmsnorm_fwd", x, w, eps=None)
    assert not both("rmsnorm_fwd", x) and not both("rmsnorm_fwd", x, w, 1e-6, True, 1) and not both("rmsnorm_fwd", x, w, weight=w) and not both("rmsnorm_fwd", x, None)
    left = []
    L._wrap.dry(left)
    try:
        with torch.device("cpu"), pytest.raises(RuntimeError, match="no CPU fallback"):
            K.rmsnorm_fwd(x, w)
        from torch.utils._python_dispatch import TorchDispatchMode

        with TorchDispatchMode(), pytest.raises(RuntimeError, match="no CPU fallback"):
            K.rmsnorm_fwd(x, w)
    finally:
        L._wrap.dry(None)
    assert left == [("left", "rmsnorm_fwd")] * 2
    with pytest.raises(RuntimeError, match="no CPU fallback"):
        K.rmsnorm_fwd(x, w)  # and a tensor that is not on the GPU


def test_results_need_no_gradient_and_know_inference_mode():
    x, w = rows(4, 16).requires_grad_(), torch.randn(16).to(B)
    calls = []
    L._wrap.dry(calls)
    try:
        y, _ = K.rmsnorm_fwd(x, w)
        with torch.inference_mode():
            z, _ = K.rmsnorm_fwd(x, w)
    finally:
        L._wrap.dry(None)
    assert [c[0] for c in calls] == ["mi355_rmsnorm_fwd"] * 2 and not y.requires_grad and not y.is_inference() and z.is_inference()
