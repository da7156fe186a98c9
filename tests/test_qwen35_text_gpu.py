"""The Qwen3.5 text stack on HIP kernels vs the CPU oracle (oracle/qwen3_5_text.py, itself
pinned to fixtures generated from the reference): kernel level first, then layers and the tiny hybrid model.
Bit-exact: index gathers.  <= 1 bf16 ulp: elementwise ops whose rounding points are reproduced.  Stated relative-L2 tolerances
elsewhere (bf16 operands, fp32 accumulation in a different order than ATen's)."""

import numpy as np
import pytest
import torch
import torch.nn.functional as F

from conftest import sub_dict
from oracle import qwen3_5_text as OT

pytestmark = pytest.mark.gpu
BF16, F32 = torch.bfloat16, torch.float32


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("needs an MI355X")


def rel_l2(a, b):
    a, b = a.double().cpu(), b.double().cpu()
    return float((a - b).norm() / (b.norm() + 1e-30))


def ulp_diff(a, b):
    """max distance in bf16 ulps between two bf16 tensors (monotone integer view)."""
    def key(t):
        i = t.cpu().contiguous().view(torch.int16).to(torch.int32)
        return torch.where(i < 0, -(i & 0x7FFF), i)
    return int((key(a) - key(b)).abs().max())


def tok_major(x):  # (b, h, s, d) -> [b*s, h*d]
    b, h, s, d = x.shape
    return x.permute(0, 2, 1, 3).reshape(b * s, h * d).contiguous()


def head_major(x2d, b, s, h):  # [b*s, h*d] -> (b, h, s, d)
    return x2d.reshape(b, s, h, -1).permute(0, 2, 1, 3)


# ------------------------------------------------------------------------------------------------- small ops
def test_zero_centered_rmsnorm_matches_fixture(golden):
    from llm_quest_amd import kernels as K
    from llm_quest_amd import kernels_q35 as Q

    t = golden("qwen35_text_tiny")
    x, scale = t["zc.x"], t["zc.scale"]
    w = Q.zc_weight(scale.cuda())
    assert torch.equal(w.cpu(), (1.0 + scale))  # bf16(1 + scale), the reference's own rounding
    y, _ = K.rmsnorm_fwd(x.reshape(-1, 64).cuda().contiguous(), w)
    assert ulp_diff(y.view(x.shape), t["zc.out"]) <= 1
    # real width
    torch.manual_seed(0)
    x = torch.randn(37, 1024).to(BF16)
    sc = (0.1 * torch.randn(1024)).to(BF16)
    y, _ = K.rmsnorm_fwd(x.cuda(), Q.zc_weight(sc.cuda()))
    assert ulp_diff(y, OT.zc_rmsnorm(x, sc)) <= 1


def test_mrope_table_is_an_exact_gather(golden):
    from llm_quest_amd import kernels_q35 as Q

    t = golden("qwen35_text_tiny")
    cos, sin, pid = t["mrope.cos"], t["mrope.sin"], t["mrope.pid"]
    ct, st = Q.mrope_table(cos.cuda(), sin.cuda(), pid.cuda(), [3, 3, 2])
    rc, rs = OT.mrope_coeffs(cos, sin, pid, [3, 3, 2])
    assert torch.equal(ct.cpu().view(2, 10, -1), rc) and torch.equal(st.cpu().view(2, 10, -1), rs)
    # real section sizes, rotation dim 64
    torch.manual_seed(1)
    cos, sin = torch.randn(512, 64), torch.randn(512, 64)
    cos[:, 32:], sin[:, 32:] = cos[:, :32], sin[:, :32]
    pid = torch.randint(0, 512, (3, 3, 41))
    ct, st = Q.mrope_table(cos.cuda(), sin.cuda(), pid.cuda(), [11, 11, 10])
    rc, rs = OT.mrope_coeffs(cos, sin, pid, [11, 11, 10])
    assert torch.equal(ct.cpu().view(3, 41, -1), rc) and torch.equal(st.cpu().view(3, 41, -1), rs)


@pytest.mark.parametrize("H,D,R,stride_mul", [(8, 256, 64, 2), (2, 256, 64, 1), (2, 32, 16, 2), (3, 128, 64, 1)])
def test_headnorm_rope_forward_backward(H, D, R, stride_mul):
    from llm_quest_amd import kernels_q35 as Q

    torch.manual_seed(2)
    b, s = 2, 19
    tokens = b * s
    hs = D * stride_mul
    proj = torch.randn(tokens, H * hs + 24).to(BF16)  # heads strided inside a wider projection
    scale = (0.2 * torch.randn(D)).to(BF16)
    cos_t, sin_t = torch.randn(tokens, R), torch.randn(tokens, R)
    cos_t[:, R // 2 :], sin_t[:, R // 2 :] = cos_t[:, : R // 2], sin_t[:, : R // 2]
    pos = torch.arange(tokens, dtype=torch.int32)
    x = torch.stack([proj[:, h * hs : h * hs + D] for h in range(H)], 1).view(b, s, H, D).transpose(1, 2)  # (b,H,s,D)

    def ref(xx, sc, dt):
        n = OT.zc_rmsnorm(xx, sc) if dt == BF16 else (xx * torch.rsqrt(xx.pow(2).mean(-1, keepdim=True) + 1e-6) * (1.0 + sc))
        c, sn = cos_t.view(b, 1, s, R).to(dt), sin_t.view(b, 1, s, R).to(dt)
        return OT.rope_partial(n, c, sn)

    want = ref(x, scale, BF16)
    dproj = proj.cuda()
    w = Q.zc_weight(scale.cuda())
    out, rstd = Q.headnorm_rope_fwd(dproj[:, : H * hs], H, D, hs, w, cos_t.cuda(), sin_t.cuda(), pos.cuda())
    got = head_major(out, b, s, H)
    assert ulp_diff(got, want) <= 1
    # backward vs fp32 autograd of the same function (bf16-rounded coefficients)
    xf = x.float().requires_grad_(True)
    sf = (1.0 + scale).float() - 1.0  # so that (1 + sf) == the bf16-rounded factor the kernel uses
    sf.requires_grad_(True)
    cb, sb = cos_t.to(BF16).float().view(b, 1, s, R), sin_t.to(BF16).float().view(b, 1, s, R)
    n = xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + 1e-6) * (1.0 + sf)
    y = OT.rope_partial(n, cb, sb)
    g = torch.randn(b, H, s, D).to(BF16)
    y.backward(g.float())
    dsrc = torch.zeros_like(dproj)
    dw = Q.headnorm_rope_bwd(dproj[:, : H * hs], H, D, hs, w, cos_t.cuda(), sin_t.cuda(), pos.cuda(), rstd, tok_major(g).cuda(), dsrc[:, : H * hs], hs)
    gx = torch.stack([dsrc.cpu()[:, h * hs : h * hs + D] for h in range(H)], 1).view(b, s, H, D).transpose(1, 2)
    assert rel_l2(gx, xf.grad) < 6e-3  # bf16 rounding of the written gradient
    assert rel_l2(dw, sf.grad) < 1e-4
    if stride_mul == 2:  # the gate halves between the heads are not touched
        for h in range(H):
            assert not dsrc.cpu()[:, h * hs + D : (h + 1) * hs].any()


@pytest.mark.parametrize("tokens,H,D,R", [(1, 1, 64, 64), (37, 3, 64, 16), (5, 1, 128, 32), (700, 5, 128, 0), (3, 3, 256, 16), (61, 2, 256, 64)])
def test_headnorm_rope_by_pieces_matches_waves(tokens, H, D, R):
    """Rows by 16-byte pieces against a wavefront a row (the same columns one element further on): sums in another order, so an element may round the other way."""
    from llm_quest_amd import kernels_q35 as Q

    torch.manual_seed(D + R)
    hs = D + 24
    src, g, w = torch.randn(tokens, H * hs).to(BF16), torch.randn(tokens, H * D).to(BF16).cuda(), (1 + 0.2 * torch.randn(D)).to(BF16).cuda()
    tab = [torch.randn(tokens + 3, R).cuda() for _ in range(2)] if R else [None, None]
    pos = torch.randint(0, tokens + 3, (tokens,), dtype=torch.int32).cuda() if R else None
    got = []
    for shift in (0, 1):
        buf = torch.cat([torch.zeros(tokens, shift, dtype=BF16), src, torch.zeros(tokens, 8 - shift, dtype=BF16)], 1).cuda()
        dbuf = torch.full_like(buf, 7.0)
        view = buf[:, shift : shift + H * hs]
        out, rstd = Q.headnorm_rope_fwd(view, H, D, hs, w, *tab, pos)
        dw = Q.headnorm_rope_bwd(view, H, D, hs, w, *tab, pos, rstd, g, dbuf[:, shift : shift + H * hs], hs)
        d = dbuf[:, shift : shift + H * hs].reshape(tokens, H, hs)
        assert bool((d[:, :, D:] == 7.0).all())
        got.append((out, rstd, d[:, :, :D], dw))
    (o0, r0, d0, w0), (o1, r1, d1, w1) = got
    assert rel_l2(r0, r1) < 1e-6 and rel_l2(w0, w1) < 1e-5
    # a normed value off by an ulp (2^-8) turns into both columns of its pair, |cos| and |sin| up to 5
    assert rel_l2(o0, o1) < 2e-3 and float((o0.float() - o1.float()).abs().max()) <= 2.0**-8 * 12 * float(o1.float().abs().max())
    assert rel_l2(d0, d1) < 1e-3 and float((d0.float() - d1.float()).abs().max()) <= 2.0**-7 * float(d1.float().abs().max())


def test_sigmoid_gate():
    from llm_quest_amd import kernels_q35 as Q

    torch.manual_seed(3)
    tokens, H, D = 45, 8, 256
    proj = torch.randn(tokens, H * 2 * D + 16).to(BF16)
    ctx = torch.randn(tokens, H * D).to(BF16)
    gate = proj[:, : H * 2 * D].view(tokens, H, 2 * D)[..., D:].reshape(tokens, H * D)
    want = ctx * torch.sigmoid(gate)
    dproj = proj.cuda()
    out = Q.sigmoid_gate_fwd(ctx.cuda(), dproj[:, D:], H, D, 2 * D)
    assert ulp_diff(out, want) <= 1
    g = torch.randn(tokens, H * D).to(BF16)
    cf, gf = ctx.float().requires_grad_(True), gate.float().requires_grad_(True)
    (cf * torch.sigmoid(gf)).backward(g.float())
    dbuf = torch.zeros_like(dproj)
    dctx = Q.sigmoid_gate_bwd(ctx.cuda(), dproj[:, D:], H, D, 2 * D, g.cuda(), dbuf[:, D:], 2 * D)
    assert rel_l2(dctx, cf.grad) < 6e-3
    dgate = dbuf.cpu()[:, : H * 2 * D].view(tokens, H, 2 * D)[..., D:].reshape(tokens, H * D)
    assert rel_l2(dgate, gf.grad) < 6e-3
    assert not dbuf.cpu()[:, : H * 2 * D].view(tokens, H, 2 * D)[..., :D].any()


def test_gdn_gates():
    from llm_quest_amd import kernels_q35 as Q

    torch.manual_seed(4)
    tokens, Hv = 333, 16
    proj = (2.0 * torch.randn(tokens, 64)).to(BF16)
    log_A = torch.log(torch.rand(Hv) * 16)
    dtb = (1.0 + 0.1 * torch.randn(Hv)).to(BF16)
    b_lin, a_lin = proj[:, 24 : 24 + Hv], proj[:, 40 : 40 + Hv]
    beta_ref = torch.sigmoid(b_lin)  # bf16
    alpha_ref = OT.alpha_factor(log_A, a_lin, dtb)  # fp32 (bf16 add, bf16 softplus)
    dproj = proj.cuda()
    beta, alpha = Q.gdn_gates_fwd(dproj[:, 24 : 24 + Hv], dproj[:, 40 : 40 + Hv], log_A.cuda(), dtb.cuda())
    assert ulp_diff(beta.to(BF16), beta_ref) <= 1 and torch.equal(beta.cpu(), beta.cpu().to(BF16).float())
    assert alpha.dtype == F32 and rel_l2(alpha, alpha_ref) < 1e-6
    # backward vs fp32 autograd
    bl, al = b_lin.float().requires_grad_(True), a_lin.float().requires_grad_(True)
    la, db = log_A.clone().requires_grad_(True), dtb.float().requires_grad_(True)
    gb, ga = torch.randn(tokens, Hv), torch.randn(tokens, Hv)
    (torch.sigmoid(bl) * gb).sum().backward()
    (OT.alpha_factor(la, al, db) * ga).sum().backward()
    dbuf = torch.zeros_like(dproj)
    dla, ddb = Q.gdn_gates_bwd(dproj[:, 24 : 24 + Hv], dproj[:, 40 : 40 + Hv], log_A.cuda(), dtb.cuda(), gb.cuda(), ga.cuda(), dbuf[:, 24 : 24 + Hv], dbuf[:, 40 : 40 + Hv])
    assert rel_l2(dbuf[:, 24 : 24 + Hv], bl.grad) < 6e-3
    assert rel_l2(dbuf[:, 40 : 40 + Hv], al.grad) < 2e-2  # softplus input / output are bf16-rounded in the forward
    assert rel_l2(dla, la.grad) < 2e-2 and rel_l2(ddb, db.grad) < 2e-2


@pytest.mark.parametrize("B,S,C", [(2, 37, 6144), (3, 5, 128), (1, 2, 64)])
def test_causal_conv_silu(B, S, C):
    from llm_quest_amd import kernels_q35 as Q

    torch.manual_seed(5)
    proj = torch.randn(B * S, C + 40).to(BF16)
    w = (0.5 * torch.randn(C, 1, 4)).to(BF16)
    x = proj[:, :C].reshape(B, S, C)
    want32 = OT.causal_depthwise_conv_silu(x.float(), w.float())
    want = OT.causal_depthwise_conv_silu(x, w)  # bf16 ATen (its accumulation order is its own)
    dproj = proj.cuda()
    y = Q.causal_conv_silu_fwd(dproj[:, :C], w.cuda(), B, S)
    assert rel_l2(y, want32.reshape(B * S, C)) < 5e-3
    assert ulp_diff(y, want.reshape(B * S, C)) <= 4
    # backward vs fp32 autograd
    xf, wf = x.float().requires_grad_(True), w.float().requires_grad_(True)
    g = torch.randn(B, S, C).to(BF16)
    OT.causal_depthwise_conv_silu(xf, wf).backward(g.float())
    dbuf = torch.zeros_like(dproj)
    dw = Q.causal_conv_silu_bwd(dproj[:, :C], w.cuda(), g.reshape(B * S, C).cuda(), dbuf[:, :C], B, S)
    assert rel_l2(dbuf[:, :C], xf.grad.reshape(B * S, C)) < 1e-2
    assert rel_l2(dw.view(C, 1, 4), wf.grad) < 1e-2
    assert not dbuf.cpu()[:, C:].any()


@pytest.mark.parametrize("B,S,C", [(1, 1, 8), (2, 3, 24), (3, 32, 2056), (1, 33, 64), (2, 35, 136), (1, 101, 8)])
def test_causal_conv_silu_backward_at_chunk_edges(B, S, C):
    """One pass over chunks of 32 tokens with the three behind them: sequences around a chunk's end and shorter than the window; against the same arithmetic (dc rounded to bf16)
    in fp64, and the same bits where dx overwrites x's or dy's rows."""
    from llm_quest_amd import kernels_q35 as Q

    torch.manual_seed(S + C)
    x, w, g = torch.randn(B * S, C + 16).to(BF16), (0.5 * torch.randn(C, 1, 4)).to(BF16), torch.randn(B * S, C).to(BF16)
    xd, gd, dx = x.cuda(), g.cuda(), torch.full((B * S, C + 8), 5.0, dtype=BF16, device="cuda")
    dw = Q.causal_conv_silu_bwd(xd[:, :C], w.cuda(), gd, dx[:, :C], B, S)
    p = torch.nn.functional.pad(x[:, :C].double().view(B, S, C), (0, 0, 3, 0))
    win = torch.stack([p[:, j : j + S] for j in range(4)], -1)  # [B, S, C, 4]
    c = (win * w.double().view(C, 4)).sum(-1).float().to(BF16).double()
    sg = torch.sigmoid(c)
    dc = (g.double().view(B, S, C) * sg * (1 + c * (1 - sg))).float().to(BF16).double()
    q = torch.nn.functional.pad(dc, (0, 0, 0, 3))
    want = sum(w.double().view(C, 4)[:, j] * q[:, 3 - j : 3 - j + S] for j in range(4))
    assert rel_l2(dx[:, :C], want.reshape(B * S, C)) < 3e-3 and rel_l2(dw.view(C, 4), (dc.unsqueeze(-1) * win).sum((0, 1))) < 1e-3  # one bf16 rounding; a rounding of dc that falls the other way
    assert bool((dx[:, C:] == 5.0).all())
    ref = dx[:, :C].clone()
    over_x, over_g = xd.clone(), gd.clone()
    Q.causal_conv_silu_bwd(over_x[:, :C], w.cuda(), gd, over_x[:, :C], B, S)
    Q.causal_conv_silu_bwd(xd[:, :C], w.cuda(), over_g, over_g, B, S)
    assert torch.equal(over_x[:, :C], ref) and torch.equal(over_g, ref)


def test_causal_conv_silu_backward_takes_scratch_only_where_it_overwrites_its_operands():
    from llm_quest_amd import kernels_q35 as Q

    rows, C = 4096, 1024
    x, g, w, dx = (torch.randn(*z, device="cuda").to(BF16) for z in ((rows, C), (rows, C), (C, 1, 4), (rows, C)))
    peak = []
    for out in (dx, x):
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        Q.causal_conv_silu_bwd(x, w, g, out, 1, rows)
        peak.append(torch.cuda.max_memory_allocated() - before)
    assert peak[1] - peak[0] == rows * C * 2 and peak[0] < rows * C * 2


def test_l2norm():
    from llm_quest_amd import kernels_q35 as Q

    torch.manual_seed(6)
    tokens, H, D = 77, 16, 128
    buf = torch.randn(tokens, H * D + 64).to(BF16)
    buf[3, :D] = 0  # a zero vector: the clamped branch
    x = buf[:, : H * D].view(tokens, H, D)
    want = OT.l2_norm(x)
    dbuf_in = buf.cuda()
    y = Q.l2norm_fwd(dbuf_in[:, : H * D], H, D)
    assert ulp_diff(y.view(tokens, H, D), want) <= 1
    xf = x.float().requires_grad_(True)
    g = torch.randn(tokens, H, D).to(BF16)
    OT.l2_norm(xf).backward(g.float())
    dx = torch.zeros_like(dbuf_in)
    Q.l2norm_bwd(dbuf_in[:, : H * D], g.reshape(tokens, H * D).cuda(), dx[:, : H * D], H, D)
    assert rel_l2(dx[:, : H * D], xf.grad.reshape(tokens, H * D)) < 6e-3


@pytest.mark.parametrize("tokens,H,D", [(1, 1, 64), (3, 5, 64), (1, 3, 128), (701, 7, 128), (33, 1, 256), (2, 3, 256)])
@pytest.mark.parametrize("shift", [0, 1])
def test_head_rows_by_pieces_and_by_waves(tokens, H, D, shift):
    """l2 norm and gated RMSNorm, forward and backward, where 8, 16 or 32 lanes take a row (columns on 16 bytes) and where a wavefront does (shift 1): each against fp64."""
    from llm_quest_amd import kernels_q35 as Q

    torch.manual_seed(D + tokens)
    W = H * D
    view = lambda a: torch.cat([torch.zeros(tokens, 8 + shift, dtype=BF16), a, torch.zeros(tokens, 16 - shift, dtype=BF16)], 1).cuda()[:, 8 + shift : 8 + shift + W]
    hold = lambda: torch.full((tokens, W + 16), 3.0, dtype=BF16, device="cuda")
    x, gate, dy, w = torch.randn(tokens, W).to(BF16), torch.randn(tokens, W).to(BF16), torch.randn(tokens, W).to(BF16), 1.0 + 0.1 * torch.randn(D)
    x[0, :D] = 0  # the clamped branch
    heads = lambda a: a.double().view(tokens, H, D)
    close = lambda a, b: bool(((a.cpu().double().view(tokens, H, D) - b).abs() <= 2.0**-8 * b.abs() + 2e-6).all())  # one bf16 rounding (2^-9) and fp32 sums of 256 terms

    y = Q.l2norm_fwd(view(x), H, D)
    inv = (1 / heads(x).norm(dim=-1, keepdim=True).float().to(BF16).clamp_min(1e-6).float()).to(BF16).double()
    assert bool(((y.cpu().double().view(tokens, H, D) - heads(x) * inv).abs() <= 2.0**-6 * (heads(x) * inv).abs()).all())  # the norm and its inverse may round the other way
    out = hold()
    Q.l2norm_bwd(view(x), dy.cuda(), out[:, shift : shift + W], H, D)
    n = heads(x).norm(dim=-1, keepdim=True)
    k3 = torch.where(n < 1e-6, 0.0, (heads(x) * heads(dy)).sum(-1, keepdim=True) / n.clamp_min(1e-6) ** 3)
    want = heads(dy) / n.clamp_min(1e-6) - heads(x) * k3
    assert bool(((out[:, shift : shift + W].cpu().double().view(tokens, H, D) - want).abs() <= 2.0**-8 * want.abs() + 2e-6 * (heads(dy).abs() / n.clamp_min(1e-6) + 1)).all())
    assert bool((out[:, shift + W :] == 3.0).all()) and bool((out[:, :shift] == 3.0).all())

    got, rstd = Q.gated_rmsnorm_fwd(x.cuda(), w.cuda(), view(gate), H, D)
    r = torch.rsqrt(heads(x).pow(2).mean(-1, keepdim=True) + 1e-6)
    g, d, wd = heads(gate), heads(dy), w.double()
    sg = torch.sigmoid(g)
    assert close(got, g * sg * heads(x) * r * wd)
    dgate = hold()
    d_o, dw = Q.gated_rmsnorm_bwd(x.cuda(), w.cuda(), view(gate), rstd, dy.cuda(), dgate[:, shift : shift + W], H, D)
    xh = heads(x) * r
    assert close(dgate[:, shift : shift + W], d * xh * wd * sg * (1 + g * (1 - sg)))
    dn = d * g * sg
    want = r * (dn * wd - xh * (dn * wd * xh).mean(-1, keepdim=True))
    assert bool(((d_o.cpu().double().view(tokens, H, D) - want).abs() <= 2.0**-8 * want.abs() + 4e-6 * r * (1 + xh.abs())).all())
    assert rel_l2(dw, (dn * xh).sum((0, 1))) < 1e-5
    assert bool((dgate[:, shift + W :] == 3.0).all()) and bool((dgate[:, :shift] == 3.0).all())


def test_gated_rmsnorm():
    from llm_quest_amd import kernels_q35 as Q
    from oracle import ops as OO

    torch.manual_seed(7)
    tokens, H, D = 91, 16, 128
    o = torch.randn(tokens, H * D).to(BF16)
    proj = torch.randn(tokens, H * D + 32).to(BF16)
    w = 1.0 + 0.1 * torch.randn(D)
    gate = proj[:, 32:]

    def ref(of, wf, gf):
        xn = of.view(tokens, H, D)
        xn = xn * torch.rsqrt(xn.pow(2).mean(-1, keepdim=True) + 1e-6) * wf
        return F.silu(gf) * xn.reshape(tokens, H * D)

    want = ref(o.float(), w, gate.float()).to(BF16)
    dproj = proj.cuda()
    out, rstd = Q.gated_rmsnorm_fwd(o.cuda(), w.cuda(), dproj[:, 32:], H, D)
    assert ulp_diff(out, want) <= 1
    of, wf, gf = o.float().requires_grad_(True), w.clone().requires_grad_(True), gate.float().requires_grad_(True)
    g = torch.randn(tokens, H * D).to(BF16)
    ref(of, wf, gf).backward(g.float())
    dbuf = torch.zeros_like(dproj)
    d_o, dw = Q.gated_rmsnorm_bwd(o.cuda(), w.cuda(), dproj[:, 32:], rstd, g.cuda(), dbuf[:, 32:], H, D)
    assert rel_l2(d_o, of.grad) < 6e-3 and rel_l2(dbuf[:, 32:], gf.grad) < 6e-3 and rel_l2(dw, wf.grad) < 1e-4


# ------------------------------------------------------------------------------------------------- gated delta rule
def _gdr_run(q, k, v, beta, alpha, go):
    """q,k: (b,hqk,s,dk) bf16; v: (b,hv,s,dv) bf16; beta/alpha (b,hv,s) fp32; go (b,hv,s,dv) fp32.  HIP forward + backward."""
    from llm_quest_amd import kernels_q35 as Q

    b, hqk, s, dk = q.shape
    hv, dv = v.shape[1], v.shape[3]
    qd, kd = tok_major(q).cuda(), tok_major(k).cuda()
    vbuf = torch.zeros(b * s, hv * dv + 16, dtype=BF16)
    vbuf[:, : hv * dv] = tok_major(v)
    vbuf = vbuf.cuda()
    be = beta.permute(0, 2, 1).reshape(b * s, hv).contiguous().cuda()
    al = alpha.permute(0, 2, 1).reshape(b * s, hv).contiguous().cuda()
    o, ck, fin = Q.gated_delta_rule_fwd(qd, kd, vbuf[:, : hv * dv], be, al, b, s, hqk, hv, dk, dv, keep=True, want_state=True)
    dvbuf = torch.zeros_like(vbuf)
    dq, dk_, dbe, dal = Q.gated_delta_rule_bwd(qd, kd, vbuf[:, : hv * dv], be, al, ck, tok_major(go.to(BF16)).cuda(), dvbuf[:, : hv * dv], b, s, hqk, hv, dk, dv)
    back = lambda t, h: head_major(t.cpu(), b, s, h)
    return (back(o, hv), fin.cpu(), back(dq, hqk), back(dk_, hqk), back(dvbuf[:, : hv * dv], hv),
            dbe.cpu().view(b, s, hv).permute(0, 2, 1), dal.cpu().view(b, s, hv).permute(0, 2, 1))


def test_gated_delta_rule_matches_reference_fixture(golden):
    t = golden("qwen35_text_tiny")
    q, k, v, beta, alpha, go = (t["gdr." + n] for n in ("q", "k", "v", "beta", "alpha", "gout"))
    o, fin, dq, dk, dv, dbeta, dalpha = _gdr_run(q, k, v, beta, alpha, go.to(BF16).float())
    assert ulp_diff(o, t["gdr.out"]) <= 1
    assert rel_l2(fin, t["gdr.state"]) < 1e-5
    # the fixture's upstream gradient is fp32; ours enters as bf16 -> bf16-level agreement
    for got, name in ((dq, "q"), (dk, "k"), (dv, "v"), (dbeta, "beta"), (dalpha, "alpha")):
        assert rel_l2(got, t["gdr.grad." + name]) < 8e-3, name


def test_gated_delta_rule_real_head_dims_three_chunks():
    torch.manual_seed(8)
    b, hqk, hv, s, dk, dv = 2, 2, 4, 150, 128, 128  # 3 checkpoint chunks, value heads share q/k heads in pairs
    q = OT.l2_norm(torch.randn(b, hqk, s, dk)).to(BF16)
    k = OT.l2_norm(torch.randn(b, hqk, s, dk)).to(BF16)
    v = torch.randn(b, hv, s, dv).to(BF16)
    beta = torch.rand(b, hv, s).to(BF16).float()
    alpha = 0.3 + 0.7 * torch.rand(b, hv, s)
    go = torch.randn(b, hv, s, dv).to(BF16).float()
    o, fin, dq, dk_, dv_, dbeta, dalpha = _gdr_run(q, k, v, beta, alpha, go)
    qf, kf, vf = (x.float().requires_grad_(True) for x in (q, k, v))
    bf_, af = beta.clone().requires_grad_(True), alpha.clone().requires_grad_(True)
    ro, rstate = OT.gated_delta_rule(qf.repeat_interleave(2, 1), kf.repeat_interleave(2, 1), vf, bf_, af)
    assert rel_l2(o, ro) < 4e-3  # bf16 rounding of the output; sums of 128 products in another order than ATen
    assert rel_l2(fin, rstate) < 1e-5
    (ro * go).sum().backward()
    assert rel_l2(dq, qf.grad) < 6e-3 and rel_l2(dk_, kf.grad) < 6e-3 and rel_l2(dv_, vf.grad) < 6e-3
    assert rel_l2(dbeta, bf_.grad) < 1e-4 and rel_l2(dalpha, af.grad) < 1e-4


# ------------------------------------------------------------------------------------------------- attention (SDPA semantics)
@pytest.mark.parametrize("B,S,Hq,Hkv,D,masked", [(2, 300, 8, 2, 256, False), (2, 173, 8, 2, 256, True), (2, 40, 2, 1, 32, True), (1, 130, 4, 2, 128, False), (1, 65, 2, 2, 64, False)])
def test_attention_generic_forward_backward(B, S, Hq, Hkv, D, masked):
    from llm_quest_amd import kernels_q35 as Q

    torch.manual_seed(9)
    q = torch.randn(B, Hq, S, D).to(BF16)
    k = torch.randn(B, Hkv, S, D).to(BF16)
    v = torch.randn(B, Hkv, S, D).to(BF16)
    am = None
    allow = torch.tril(torch.ones(S, S, dtype=torch.bool))
    if masked:
        am = torch.ones(B, S, dtype=torch.bool)
        am[0, S - 7 :] = False
        am[B - 1, S // 2 : S // 2 + 3] = False  # upstream ORs ~attn_mask into the allow mask: these keys become visible to all
        allow = allow.view(1, 1, S, S) | ~am.view(B, 1, 1, S)
    qf, kf, vf = (x.float().requires_grad_(True) for x in (q, k, v))
    ref = F.scaled_dot_product_attention(qf, kf, vf, attn_mask=allow, enable_gqa=True)
    go = torch.randn(B, Hq, S, D).to(BF16)
    ref.backward(go.float())
    qd, kd, vd = tok_major(q).cuda(), tok_major(k).cuda(), tok_major(v).cuda()
    km = None if am is None else am.to(torch.uint8).cuda()
    o, lse = Q.attn_generic_fwd(qd, kd, vd, B, S, Hq, Hkv, D, key_mask=km)
    assert rel_l2(head_major(o, B, S, Hq), ref) < 6e-3
    dq, dk, dv = torch.empty_like(qd), torch.empty_like(kd), torch.empty_like(vd)
    Q.attn_generic_bwd(qd, kd, vd, o, tok_major(go).cuda(), lse, B, S, Hq, Hkv, D, dq, dk, dv, key_mask=km)
    assert rel_l2(head_major(dq, B, S, Hq), qf.grad) < 1e-2
    assert rel_l2(head_major(dk, B, S, Hkv), kf.grad) < 1e-2
    assert rel_l2(head_major(dv, B, S, Hkv), vf.grad) < 1e-2
    # determinism
    o2, _ = Q.attn_generic_fwd(qd, kd, vd, B, S, Hq, Hkv, D, key_mask=km)
    assert torch.equal(o, o2)


# ------------------------------------------------------------------------------------------------- layers and the tiny hybrid model
from oracle.gen_golden import TINY_Q35_TEXT


def _fp32_twin(sd):
    return {k: (v.float() if v.dtype == BF16 else v) for k, v in sd.items()}


def _twin_forward_backward(sd, cfg, ids, am, pid, gout):
    """fp32 twin of the reference model (same weights upcast) through the oracle, with autograd: logits + parameter gradients."""
    tw = _fp32_twin(sd)
    leaves = {k: v.clone().requires_grad_(True) for k, v in tw.items() if v.dtype == F32 and k not in ("cos", "sin")}
    full = {**tw, **leaves}
    full["mask"] = sd["mask"].bool()
    if cfg["tie_embeddings"]:
        full["out_head.weight"] = full["emb_dict.weight"]
    logits = OT.text_model_forward(full, cfg, x=ids, attn_mask=am, position_ids=pid)
    (logits * gout).sum().backward()
    return logits.detach(), {k: v.grad for k, v in leaves.items() if v.grad is not None}


def test_tiny_hybrid_model_forward_backward_vs_reference(golden):
    from llm_quest_amd.qwen.qwen3_5.qwen3_5_text_model import Qwen3_5TextModel

    t = golden("qwen35_text_tiny")
    cfg = {**TINY_Q35_TEXT, "dtype": BF16}
    sd = sub_dict(t, "txt.bf16.sd.")
    ids, am, pid, gout = t["txt.ids"], t["txt.attn_mask"].bool(), t["txt.pid"], t["txt.gout"]
    m = Qwen3_5TextModel(cfg)
    assert set(m.state_dict()) == set(sd)
    m.load_state_dict({k: (v.bool() if k == "mask" else v) for k, v in sd.items()})
    m = m.cuda().train()
    twin_logits, twin_grads = _twin_forward_backward(sd, cfg, ids, am, pid, gout)
    logits = m(ids.cuda(), attn_mask=am.cuda(), position_ids=pid.cuda())
    assert logits.dtype == BF16 and logits.shape == t["txt.bf16.logits"].shape
    floor = rel_l2(t["txt.bf16.logits"], twin_logits)  # the reference's own bf16 noise vs its fp32 twin
    mine = rel_l2(logits, twin_logits)
    assert mine <= 1.5 * floor + 1e-3, f"logits vs fp32 twin {mine:.3e}, reference floor {floor:.3e}"
    assert rel_l2(logits, t["txt.bf16.logits"]) <= 2.0 * floor + 1e-3
    (logits.float() * gout.cuda()).sum().backward()
    report, bad = [], []
    for name, p in m.named_parameters():
        if name == "out_head.weight":
            continue
        ref = t["txt.bf16.grad." + name]
        assert p.grad is not None and p.grad.dtype == ref.dtype and p.grad.shape == ref.shape, name
        tg = twin_grads[name]
        floor_g = rel_l2(ref, tg)
        mine_g = rel_l2(p.grad, tg)
        # gate parameters with a handful of elements (log_A, dt_bias, w_alpha: 4 value heads here) carry the bf16 rounding of
        # softplus / sigmoid in both implementations; their noise is not averaged over many elements, hence the wider factor
        factor = 2.5 if ref.numel() <= 256 and ("log_A" in name or "dt_bias" in name or "w_alpha" in name or "w_beta" in name) else 1.5
        report.append(f"{name}: mine {mine_g:.3e} floor {floor_g:.3e}")
        if mine_g > factor * floor_g + (0.0 if floor_g >= 1e-2 else 2e-3):  # no additive slack where the reference's own noise is >= 1e-2
            bad.append(report[-1])
    print("\n".join(report))
    assert not bad, bad
    # text-only path (no position ids, no mask): 1-D RoPE through GatedAttention.forward
    with torch.no_grad():
        lt = m.eval()(ids.cuda())
    tw = _fp32_twin(sd)
    tw["mask"] = sd["mask"].bool()
    tw["out_head.weight"] = tw["emb_dict.weight"]
    twin_t = OT.text_model_forward(tw, cfg, x=ids)
    floor_t = rel_l2(t["txt.bf16.logits_text_only"], twin_t)
    assert rel_l2(lt, twin_t) <= 1.5 * floor_t + 1e-3


def _layer_cfg():
    return dict(emb_dim=1024, hidden_dim=3584, n_heads=8, num_kv_groups=2, head_dim=256, rope_base=10_000_000, partial_rope_factor=0.25,
                context_length=256, linear_num_qk_heads=16, linear_num_value_heads=16, linear_qk_head_dim=128, linear_value_head_dim=128,
                linear_conv_kernel_size=4, p_dropout=0.0, training=False, mrope_section=[11, 11, 10], dtype=BF16, linear_sdpa_ratio=4,
                vocab_size=512, n_layers=1, tie_embeddings=True)


@pytest.mark.parametrize("kind", ["gdn", "attention"])
def test_real_width_blocks_vs_oracle(kind):
    """One Qwen3.5-0.8B-sized block (d 1024, GDN 16x128 heads / gated attention 8x256 heads over 2 kv groups, ffn 3584) forward and
    backward vs the oracle: bf16 oracle for the output (reference arithmetic), fp32 twin for gradients."""
    from llm_quest_amd.common.buffers import GlobalBuffers
    from llm_quest_amd.qwen.qwen3_5.qwen3_5_text_model import Qwen3_5TransformerBlock

    torch.manual_seed(11)
    cfg = _layer_cfg()
    layer_idx = 0 if kind == "gdn" else 3
    blk = Qwen3_5TransformerBlock(cfg, layer_idx)
    with torch.no_grad():
        for n_, p_ in blk.named_parameters():
            if n_.endswith("scale") or n_.endswith("post_norm.weight") or n_.endswith("dt_bias"):
                p_.add_((0.1 * torch.randn(p_.shape)).to(p_.dtype))
    sd = {"trf_blocks.0." + k: v.detach().clone() for k, v in blk.state_dict().items()}
    b, s = 2, 75
    x = torch.randn(b, s, 1024).to(BF16)
    am = torch.ones(b, s, dtype=torch.bool)
    am[1, 70:] = False
    pid = torch.arange(s).view(1, 1, s).repeat(3, b, 1)
    pid[1, :, 10:30] = 10 + torch.arange(20) // 5
    pid[2, :, 10:30] = 10 + torch.arange(20) % 5
    cos, sin = GlobalBuffers.get_rope_params(256, cfg["rope_base"], 256, rotation_factor=0.25)
    allow = ~GlobalBuffers.get_causal_mask(256)
    ocfg = {**cfg, "linear_sdpa_ratio": 1 if kind == "attention" else 4}  # oracle decides the layer kind from the index
    want = OT.block(sd, "trf_blocks.0.", ocfg, 0, x, allow, cos, sin, pid, am)
    tw = {k: (v.float().requires_grad_(True) if v.is_floating_point() else v) for k, v in sd.items()}
    xf = x.float().requires_grad_(True)
    ref32 = OT.block(tw, "trf_blocks.0.", ocfg, 0, xf, allow, cos, sin, pid, am)
    g = torch.randn(b, s, 1024).to(BF16)
    ref32.backward(g.float())
    blk = blk.cuda().train()
    xd = x.cuda().requires_grad_(True)
    y = blk(xd, allow.cuda(), cos.cuda(), sin.cuda(), pid.cuda(), am.cuda())
    floor = rel_l2(want, ref32)
    assert rel_l2(y, ref32) <= 1.5 * floor + 1e-3, (rel_l2(y, ref32), floor)
    y.backward(g.cuda())
    # gradients on the floor rule: the oracle's bf16 run (the reference's arithmetic) against its fp32 twin sets the bar for every tensor
    low = {k: (v.detach().clone().requires_grad_(True) if v.is_floating_point() else v) for k, v in sd.items()}
    xl = x.clone().requires_grad_(True)
    OT.block(low, "trf_blocks.0.", ocfg, 0, xl, allow, cos, sin, pid, am).backward(g)
    floor_x = rel_l2(xl.grad, xf.grad)
    assert rel_l2(xd.grad, xf.grad) <= 1.5 * floor_x + (0.0 if floor_x >= 1e-2 else 2e-3), (rel_l2(xd.grad, xf.grad), floor_x)
    for name, p in blk.named_parameters():
        tg = tw["trf_blocks.0." + name].grad
        assert p.grad is not None, name
        floor_g = rel_l2(low["trf_blocks.0." + name].grad, tg)
        mine_g = rel_l2(p.grad, tg)
        # the handful-of-elements gate parameters carry un-averaged bf16 rounding of softplus / sigmoid in both implementations (see the tiny-model test)
        few = tg.numel() <= 256 and any(s_ in name for s_ in ("log_A", "dt_bias"))
        assert mine_g <= (2.5 if few else 1.5) * floor_g + (0.0 if floor_g >= 1e-2 else 2e-3), f"{name}: mine {mine_g:.3e}, oracle bf16 floor {floor_g:.3e}"


def test_functional_gated_delta_rule_has_the_reference_signature(golden):
    from llm_quest_amd.qwen.qwen3_next.qwen3_next_attention import gated_delta_rule

    t = golden("qwen35_text_tiny")
    q, k, v, beta, alpha = (t["gdr." + n].cuda().requires_grad_(True) for n in ("q", "k", "v", "beta", "alpha"))
    o, state = gated_delta_rule(q, k, v, beta, alpha)
    assert o.dtype == BF16 and ulp_diff(o, t["gdr.out"]) <= 1 and rel_l2(state, t["gdr.state"]) < 1e-5
    (o.float() * t["gdr.gout"].cuda()).sum().backward()
    for ten, name in ((q, "q"), (k, "k"), (v, "v"), (beta, "beta"), (alpha, "alpha")):
        assert ten.grad.dtype == t["gdr.grad." + name].dtype and rel_l2(ten.grad, t["gdr.grad." + name]) < 8e-3, name


def test_functional_gated_delta_rule_carries_a_previous_state(golden):
    """prev_state (reference :103-159): running the sequence in two pieces, the second from the first piece's state, gives the one-piece result;
    prev_state itself is left untouched (training through it: test_gated_delta_rule_trains_through_a_carried_state)."""
    from llm_quest_amd.qwen.qwen3_next.qwen3_next_attention import gated_delta_rule

    t = golden("qwen35_text_tiny")
    q, k, v, beta, alpha = (t["gdr." + n].cuda() for n in ("q", "k", "v", "beta", "alpha"))
    s = q.shape[2]
    cut = s // 2
    with torch.no_grad():
        o_all, st_all = gated_delta_rule(q, k, v, beta, alpha)
        o1, st1 = gated_delta_rule(q[:, :, :cut], k[:, :, :cut], v[:, :, :cut], beta[:, :, :cut], alpha[:, :, :cut])
        keep = st1.clone()
        o2, st2 = gated_delta_rule(q[:, :, cut:], k[:, :, cut:], v[:, :, cut:], beta[:, :, cut:], alpha[:, :, cut:], prev_state=st1)
    assert torch.equal(st1, keep), "prev_state must not be modified"
    assert torch.equal(o1, o_all[:, :, :cut]) and ulp_diff(o2, o_all[:, :, cut:].contiguous()) <= 1 and rel_l2(st2, st_all) < 1e-6
    assert ulp_diff(torch.cat((o1, o2), 2), t["gdr.out"]) <= 1 and rel_l2(st2, t["gdr.state"]) < 1e-5
    o3, st3 = gated_delta_rule(q[:, :, cut:].clone().requires_grad_(True), k[:, :, cut:], v[:, :, cut:], beta[:, :, cut:], alpha[:, :, cut:], prev_state=st1)
    assert torch.equal(o3.detach(), o2) and torch.equal(st3.detach(), st2) and torch.equal(st1, keep), "the differentiable path computes the same forward"


@pytest.mark.parametrize("s", [64, 65, 130])
def test_functional_gated_delta_rule_takes_any_decay_and_any_key(s):
    """The public entry with a carried state, heads of 128 | 128 and whole chunks of tokens, on operands that no layer makes: decays below and at zero, keys that are not unit
    vectors.  With and without gradients it is one recurrence (the same bits), and that of fp64: the state is fp32 (128 products a step, some 2^-24 sqrt(s) each), the output is
    rounded to bf16 (2^-9)."""
    from llm_quest_amd.qwen.qwen3_next.qwen3_next_attention import gated_delta_rule

    g = torch.Generator().manual_seed(s)
    b, h, D = 1, 2, 128
    q, v = (torch.randn(b, h, s, D, generator=g).to(BF16) for _ in range(2))
    k = (torch.randn(b, h, s, D, generator=g) * (0.7 / D**0.5)).to(BF16)
    beta, alpha = torch.sigmoid(torch.randn(b, h, s, generator=g)), 0.5 + 0.5 * torch.rand(b, h, s, generator=g)
    alpha[..., ::7] *= -1.0
    alpha[..., 5::31] = 0.0
    s0 = torch.randn(b, h, D, D, generator=g)
    st, outs = s0.double(), []
    for t in range(s):
        kt, a = k[:, :, t].double(), alpha[:, :, t, None, None].double()
        st = st * a
        u = beta[:, :, t, None].double() * (v[:, :, t].double() - (st * kt[:, :, None, :]).sum(-1))
        st = st + u[..., None] * kt[:, :, None, :]
        outs.append((st * q[:, :, t].double()[:, :, None, :]).sum(-1) / D**0.5)
    ref = torch.stack(outs, 2)
    with torch.no_grad():
        o, fin = gated_delta_rule(q.cuda(), k.cuda(), v.cuda(), beta.cuda(), alpha.cuda(), prev_state=s0.cuda())
    o2, fin2 = gated_delta_rule(q.cuda().requires_grad_(True), k.cuda(), v.cuda(), beta.cuda(), alpha.cuda(), prev_state=s0.cuda())
    assert torch.equal(o, o2.detach()) and torch.equal(fin, fin2.detach())
    assert rel_l2(o.float(), ref.float()) < 4e-3 and rel_l2(fin, st.float()) < 1e-5


def test_text_model_loss_path_and_determinism():
    """forward_hidden + lm_loss == CE of forward()'s logits; two identical steps give bit-identical gradients."""
    from llm_quest_amd.qwen.qwen3_5.qwen3_5_text_model import Qwen3_5TextModel

    torch.manual_seed(12)
    cfg = {**TINY_Q35_TEXT, "dtype": BF16}
    m = Qwen3_5TextModel(cfg).cuda().train()
    ids = torch.randint(0, 256, (3, 33)).cuda()
    tgt = torch.randint(0, 256, (3, 33)).cuda()

    def step():
        m.zero_grad(set_to_none=True)
        h = m.forward_hidden(ids)
        loss = m.lm_loss(h.reshape(-1, h.shape[-1]), tgt)
        loss.backward()
        return loss.detach().clone(), {n: p.grad.detach().clone() for n, p in m.named_parameters() if n != "out_head.weight"}

    l1, g1 = step()
    l2, g2 = step()
    assert torch.equal(l1, l2) and all(torch.equal(g1[n], g2[n]) for n in g1)
    with torch.no_grad():
        logits = m(ids)
    ref = F.cross_entropy(logits.float().flatten(0, 1), tgt.flatten())
    assert abs(float(l1) - float(ref)) / float(ref) < 1e-3


def test_qwen35_vlm_composes_vision_scatter_mrope_and_text_stack():
    """Qwen3_5VLM.forward == text model on (scatter(emb, vision tower), 3-D position ids): every piece is pinned on its own above
    and in test_qwen35_gpu.py; this checks the composition, bit for bit, and that a loss reaches every parameter."""
    from oracle.gen_golden import TINY_Q35_VISION
    from llm_quest_amd.qwen.qwen3_5.qwen3_5_vlm_model import Qwen3_5VLM, fuse_vision_embeddings

    torch.manual_seed(13)
    cfg = {**TINY_Q35_TEXT, **TINY_Q35_VISION, "dtype": BF16, "emb_dim": 128, "llm_d_in": 128, "image_token_id": 255, "n_heads": 2, "head_dim": 32}
    vlm = Qwen3_5VLM(cfg).cuda().train()
    n_img = (4 // 2) * (4 // 2) * (4 // 2)  # frames/2 x (32/8/2)^2 merged rows
    ids = torch.randint(0, 250, (2, 30))
    ids[:, 5 : 5 + n_img] = 255
    pix = torch.randn(2, 3, 4, 32, 32)
    logits = vlm(ids.cuda(), image_pixels=pix.cuda())
    assert logits.shape == (2, 30, 256) and logits.dtype == BF16
    lm = vlm.language_model
    with torch.no_grad():
        emb = fuse_vision_embeddings(lm.emb_dict(ids.cuda()), (ids == 255).cuda(), vlm.vision_model(pix.cuda()))
        pos = vlm.compute_3d_position_ids(ids.cuda(), vlm.get_feeds_3d_shape(pix.cuda()))
        manual = lm(inputs_embs=emb, position_ids=pos)
    assert torch.equal(logits.detach(), manual)
    F.cross_entropy(logits.float().flatten(0, 1), torch.randint(0, 256, (60,)).cuda()).backward()
    for name, p in vlm.named_parameters():
        if name.endswith("out_head.weight"):
            continue
        assert p.grad is not None and torch.isfinite(p.grad.float()).all(), name


def test_rccl_gradsync_qwen35_single_rank():
    """The RCCL path of config 5 on one GPU (1-rank 'nccl' group, GradSync forced on): block arenas during backward, the embedding arena
    and the coalesced bucket of stand-alone parameters (fp32 GDN parameters, the fp32 vision tower) in finish_step.  Gradients unchanged."""
    import os

    import torch.distributed as dist

    from oracle.gen_golden import TINY_Q35_VISION
    from llm_quest_amd import ddp
    from llm_quest_amd.qwen.qwen3_5.qwen3_5_vlm_model import Qwen3_5VLM

    torch.manual_seed(14)
    cfg = {**TINY_Q35_TEXT, **TINY_Q35_VISION, "dtype": BF16, "emb_dim": 128, "llm_d_in": 128, "image_token_id": 255, "n_heads": 2, "head_dim": 32}
    vlm = Qwen3_5VLM(cfg).cuda().train()
    ids = torch.randint(0, 250, (2, 30))
    ids[:, 5:13] = 255
    pix = torch.randn(2, 3, 4, 32, 32).cuda()
    tgt = torch.randint(0, 256, (60,)).cuda()

    def loss_fn():
        vlm.zero_grad(set_to_none=True)
        return F.cross_entropy(vlm(ids.cuda(), image_pixels=pix).float().flatten(0, 1), tgt)

    loss_fn().backward()
    ref = {n: p.grad.float().clone() for n, p in vlm.named_parameters() if p.grad is not None}
    os.environ.update(MASTER_ADDR="127.0.0.1", MASTER_PORT="29533")
    dist.init_process_group("nccl", rank=0, world_size=1, device_id=torch.device("cuda", 0))
    try:
        sync = ddp.sync_for_qwen35(vlm)
        assert len(sync.tail_params) > 0 and any(p.dtype == F32 for p in sync.tail_params)
        sync.enabled = True
        sync.broadcast_parameters([vlm])
        loss = loss_fn()
        sync.begin_step()
        loss.backward()
        sync.finish_step()
        torch.cuda.synchronize()
        assert len(sync._done) == len(vlm.language_model.trf_blocks) + 1
        for n, p in vlm.named_parameters():
            if n in ref:  # two backward passes: fp32 atomics (bias column sums, embedding scatter) may order differently; a broken sync is O(1)
                assert rel_l2(p.grad, ref[n]) < 1e-3, n
    finally:
        dist.destroy_process_group()
        for m in vlm.language_model.trf_blocks:
            object.__setattr__(m, "_grad_ready", None)


def test_gated_attention_with_attention_dropout_given_the_mask():
    """``GatedAttention`` with ``p_dropout`` > 0 under ``training`` (reference qwen3_next_attention.py:181,245-253: SDPA's ``dropout_p``): the weights are
    dropped inside the attention kernels by Philox masks that the backward regenerates.  Output and every gradient against the oracle's fp32 twin
    evaluated with the SAME mask (oracle/dropout.py); a repeat with the same (seed, offset) is bit-identical, another offset is not; the same on a padded
    batch (padding mask + dropout in one SDPA call: mi355_attn_generic_dropout_fwd / _bwd)."""
    from llm_quest_amd import rng
    from llm_quest_amd.common.buffers import GlobalBuffers
    from llm_quest_amd.qwen.qwen3_next.qwen3_next_attention import GatedAttention
    from oracle import dropout as OD

    torch.manual_seed(21)
    p, seed = 0.2, 4242
    cfg = dict(emb_dim=64, n_heads=2, num_kv_groups=1, head_dim=32, rope_base=10_000, partial_rope_factor=0.5, context_length=64, dtype=BF16,
               p_dropout=p, training=True, mrope_section=[3, 3, 2])
    att = GatedAttention(cfg)
    assert att.p_dropout == p and GatedAttention({**cfg, "training": False}).p_dropout == 0.0
    with torch.no_grad():
        for n_, p_ in att.named_parameters():
            if n_.endswith("scale"):
                p_.add_((0.1 * torch.randn(p_.shape)).to(p_.dtype))
    sd = {"a." + k: v.detach().clone() for k, v in att.state_dict().items()}
    b, s = 2, 21
    x = torch.randn(b, s, 64).to(BF16)
    g = torch.randn(b, s, 64).to(BF16)
    cos, sin = GlobalBuffers.get_rope_params(64, cfg["rope_base"], 32, rotation_factor=0.5)
    allow = ~GlobalBuffers.get_causal_mask(64)
    att = att.cuda().train()

    def run(offset):
        rng.manual(seed, offset)
        try:
            xd = x.cuda().requires_grad_(True)
            for p_ in att.parameters():
                p_.grad = None
            y = att(xd, allow.cuda(), cos.cuda(), sin.cuda())
            y.backward(g.cuda())
        finally:
            rng.follow_torch()
        return y.detach(), xd.grad.clone(), {n_: p_.grad.detach().float().clone() for n_, p_ in att.named_parameters()}

    y, dx, grads = run(0)
    y2, dx2, _ = run(0)
    y3, _, _ = run(1)
    assert torch.equal(y, y2) and torch.equal(dx, dx2) and not torch.equal(y, y3)
    mul = OD.attention_multiplier(b, 2, s, p, seed, 0)
    tw = {k: (v.float().requires_grad_(True) if v.is_floating_point() else v) for k, v in sd.items()}
    xf = x.float().requires_grad_(True)
    ref = OT.gated_attention(tw, "a.", cfg, xf, allow, cos, sin, None, None, att_mul=mul)
    ref.backward(g.float())
    assert rel_l2(y, ref) < 2e-2, rel_l2(y, ref)
    assert rel_l2(ref, OT.gated_attention(tw, "a.", cfg, xf, allow, cos, sin, None, None)) > 5e-2  # the masks really acted
    assert rel_l2(dx, xf.grad) < 3e-2, rel_l2(dx, xf.grad)
    for n_, gr in grads.items():
        assert rel_l2(gr, tw["a." + n_].grad) < 4e-2, (n_, rel_l2(gr, tw["a." + n_].grad))
    # ... and on a padded batch (SDPA gets the padding mask AND dropout_p, qwen3_next_attention.py:240-253): the same masks over the quirk-mask kernels
    am = torch.ones(b, s, dtype=torch.bool)
    am[0, 15:] = False

    def run_padded(offset):
        rng.manual(seed, offset)
        try:
            xd = x.cuda().requires_grad_(True)
            for p_ in att.parameters():
                p_.grad = None
            y_ = att(xd, allow.cuda(), cos.cuda(), sin.cuda(), attn_mask=am.cuda())
            y_.backward(g.cuda())
        finally:
            rng.follow_torch()
        return y_.detach(), xd.grad.clone(), {n_: p_.grad.detach().float().clone() for n_, p_ in att.named_parameters()}

    yp, dxp, gp = run_padded(0)
    yp2, dxp2, _ = run_padded(0)
    assert torch.equal(yp, yp2) and torch.equal(dxp, dxp2) and not torch.equal(yp, y)
    tw = {k: (v.float().requires_grad_(True) if v.is_floating_point() else v) for k, v in sd.items()}
    xf = x.float().requires_grad_(True)
    refp = OT.gated_attention(tw, "a.", cfg, xf, allow, cos, sin, None, am, att_mul=mul)
    refp.backward(g.float())
    assert rel_l2(yp, refp) < 2e-2, rel_l2(yp, refp)
    assert rel_l2(refp, OT.gated_attention(tw, "a.", cfg, xf, allow, cos, sin, None, am)) > 5e-2
    assert rel_l2(dxp, xf.grad) < 3e-2, rel_l2(dxp, xf.grad)
    for n_, gr in gp.items():
        assert rel_l2(gr, tw["a." + n_].grad) < 4e-2, (n_, rel_l2(gr, tw["a." + n_].grad))


@pytest.mark.parametrize("dk,dv,s1,s2", [(16, 16, 12, 9), (128, 128, 21, 20)])
def test_gated_delta_rule_trains_through_a_carried_state(dk, dv, s1, s2):
    """``gated_delta_rule(..., prev_state)`` under autograd (reference qwen3_next_attention.py:103-159: the recurrence simply starts from ``prev_state`` and
    returns the last state, both differentiable): a sequence cut in two -- the second call starts from the first one's state -- must give the gradients
    of the uncut sequence (the backward of the second half leaves d(prev_state), the backward of the first half starts from it), and both must match the
    oracle's recurrence under fp32 autograd, including the gradient of a carried-in state and of a loss on the returned state."""
    from llm_quest_amd.qwen.qwen3_next.qwen3_next_attention import gated_delta_rule

    torch.manual_seed(31)
    b, h, s = 2, 4, s1 + s2
    nrm = lambda t: torch.nn.functional.normalize(t, dim=-1)
    q, k = nrm(torch.randn(b, h, s, dk)).to(BF16), nrm(torch.randn(b, h, s, dk)).to(BF16)
    v = torch.randn(b, h, s, dv).to(BF16)
    beta = torch.rand(b, h, s)
    alpha = 0.5 + 0.5 * torch.rand(b, h, s)
    s0 = 0.1 * torch.randn(b, h, dv, dk)
    go = torch.randn(b, h, s, dv)
    gs = 0.1 * torch.randn(b, h, dv, dk)

    # oracle: the recurrence in fp32 autograd, from the carried-in state
    ins = [t.clone().float().requires_grad_(True) for t in (q, k, v, beta, alpha, s0)]
    qf, kf, vf, bf, af, sf = ins
    st, outs = sf, []
    for t in range(s):
        st = af[:, :, t, None, None] * st
        u = bf[:, :, t, None] * (vf[:, :, t] - (st * kf[:, :, t, None, :]).sum(-1))
        st = st + u[..., None] * kf[:, :, t, None, :]
        outs.append((st * (qf[:, :, t, None, :] * dk ** -0.5)).sum(-1))
    o_ref = torch.stack(outs, dim=2)
    ((o_ref * go).sum() + (st * gs).sum()).backward()

    def leaves():
        return [t.clone().cuda().requires_grad_(True) for t in (q, k, v, beta, alpha, s0)]

    # one call from the carried-in state
    a = leaves()
    o1, f1 = gated_delta_rule(*a[:5], prev_state=a[5])
    ((o1.float() * go.cuda()).sum() + (f1 * gs.cuda()).sum()).backward()
    assert rel_l2(o1, o_ref) < 1e-2 and rel_l2(f1, st) < 2e-3
    for name, mine, ref in zip(("q", "k", "v", "beta", "alpha", "prev_state"), a, ins):
        assert mine.grad is not None, name
        assert rel_l2(mine.grad, ref.grad) < 1.5e-2, (name, rel_l2(mine.grad, ref.grad))
    # the same sequence cut in two: the state gradient crosses the cut
    c = leaves()
    cut = lambda t, lo, hi: t[:, :, lo:hi]
    oa, fa = gated_delta_rule(*(cut(t, 0, s1) for t in c[:5]), prev_state=c[5])
    ob, fb = gated_delta_rule(*(cut(t, s1, s) for t in c[:5]), prev_state=fa)
    ((torch.cat([oa, ob], dim=2).float() * go.cuda()).sum() + (fb * gs.cuda()).sum()).backward()
    assert torch.equal(torch.cat([oa, ob], dim=2), o1) or rel_l2(torch.cat([oa, ob], dim=2), o1) < 2e-3
    for name, two, one in zip(("q", "k", "v", "beta", "alpha", "prev_state"), c, a):
        assert rel_l2(two.grad, one.grad) < 6e-3, (name, rel_l2(two.grad, one.grad))


# ------------------------------------------------------------------------------------------------- the chunked kernels of the gated delta rule
@pytest.mark.parametrize("b,hqk,hv,s,decay", [(1, 1, 1, 64, "mix"), (2, 1, 2, 65, "mix"), (1, 2, 2, 127, "slow"), (1, 1, 3, 128, "tiny"), (2, 2, 2, 200, "zero"), (1, 1, 1, 333, "keys")])
def test_chunked_gated_delta_rule_matches_the_token_by_token_kernels(b, hqk, hv, s, decay):
    """csrc/gdr_chunk.hip against the sequential kernels on the same operands (one chunk, chunks with a remainder, shared q / k heads; decays near one, far below fp32's
    resolution of their sums, and exactly zero; nearly parallel keys), carried-in state and its gradient included.  bf16 results: a rounding flips where two fp32 sums
    straddle a boundary (2^-9 of few elements); fp32 results: both sides are sums of 64 ... 128 fp32 products behind at most 64 steps of substitution."""
    from llm_quest_amd import kernels_q35 as Q

    g = torch.Generator().manual_seed(s + hv)
    D = 128
    keys = torch.randn(b, s, hqk, D, generator=g) + (3.0 if decay == "keys" else 0.0)
    q = torch.nn.functional.normalize(torch.randn(b, s, hqk, D, generator=g), dim=-1).to(BF16).reshape(b * s, -1).cuda()
    k = torch.nn.functional.normalize(keys, dim=-1).to(BF16).reshape(b * s, -1).cuda()
    wide = torch.randn(b * s, hv * D + 8, generator=g).to(BF16).cuda()
    v = wide[:, : hv * D]
    be = torch.sigmoid(torch.randn(b * s, hv, generator=g)).cuda()
    rate = {"slow": -9.0, "tiny": 2.5}.get(decay, -3.0)
    al = torch.exp(-torch.exp(rate + 2.0 * torch.rand(b * s, hv, generator=g))).cuda()
    if decay == "zero":
        al[::7] = 0.0
    go = torch.randn(b * s, hv * D, generator=g).to(BF16).cuda()
    s0, gs = (0.1 * torch.randn(b, hv, D, D, generator=g)).cuda(), (0.1 * torch.randn(b, hv, D, D, generator=g)).cuda()
    out = []
    for chunked in (False, None):
        assert Q.gdr_chunked(v, s, D, D)
        o, ck, fin = Q.gated_delta_rule_fwd(q, k, v, be, al, b, s, hqk, hv, D, D, state=s0.clone(), chunked=chunked)
        assert (ck.dim() == 1) == (chunked is None)
        dv = torch.zeros_like(wide)
        res = Q.gated_delta_rule_bwd(q, k, v, be, al, ck, go, dv[:, : hv * D], b, s, hqk, hv, D, D, d_final=gs, want_d_initial=True)
        assert bool((dv[:, hv * D :] == 0).all())
        o2, ck2, fin2 = Q.gated_delta_rule_fwd(q, k, v, be, al, b, s, hqk, hv, D, D, keep=False, state=s0.clone(), chunked=chunked)
        assert ck2 is None and torch.equal(o, o2) and torch.equal(fin, fin2)
        out.append((o, res[0], res[1], dv[:, : hv * D], fin, res[2], res[3], res[4]))
    for i, (one, two) in enumerate(zip(*out)):
        if i == 6 and decay == "zero":  # d(alpha) where alpha is zero: the sums that span such a token hold alpha itself (as 1e-30), its factor at fp32's lower end
            keep = al > 0
            one, two = one[keep], two[keep]
        assert bool(torch.isfinite(two.float()).all()) and rel_l2(two, one) < (1e-3 if i < 4 else 2e-6), (i, rel_l2(two, one))


@pytest.mark.parametrize("b,hqk,hv,s,decay", [(1, 1, 2, 64, "mix"), (2, 2, 2, 200, "mix"), (1, 1, 1, 333, "slow"), (1, 2, 2, 130, "tiny"), (1, 1, 2, 190, "zero"), (1, 2, 2, 128, "keys")])
def test_chunked_gated_delta_rule_is_as_near_to_fp64_as_the_token_by_token_kernels(b, hqk, hv, s, decay):
    """Forward and backward of both sets of kernels against the recurrence in fp64 and its autograd.  bf16 results: the rounding to bf16 is all that shows, so the two distances are the
    same (1 % beside it).  fp32 results: chains of 32 ... 128 fp32 sums, each rounding at most 2^-24 of a partial sum, some behind 63 steps of substitution: 1e-6 holds
    sqrt(128) of them and the amplification of nearly parallel keys.  ``zero``: decays and betas of exactly zero (they count as 1e-30)."""
    from llm_quest_amd import kernels_q35 as Q

    g = torch.Generator().manual_seed(3 * s + hv)
    D = 128
    keys = torch.randn(b, s, hqk, D, generator=g) + (3.0 if decay == "keys" else 0.0)
    q = torch.nn.functional.normalize(torch.randn(b, s, hqk, D, generator=g), dim=-1).to(BF16).reshape(b * s, -1).cuda()
    k = torch.nn.functional.normalize(keys, dim=-1).to(BF16).reshape(b * s, -1).cuda()
    v, go = (torch.randn(b * s, hv * D, generator=g).to(BF16).cuda() for _ in range(2))
    be = torch.sigmoid(torch.randn(b * s, hv, generator=g)).cuda()
    al = torch.exp(-torch.exp({"slow": -9.0, "tiny": 1.0}.get(decay, -3.0) + 2.0 * torch.rand(b * s, hv, generator=g))).cuda()
    if decay == "zero":
        al[5::9], be[3::11] = 0.0, 0.0
    s0, gs = ((0.1 * torch.randn(b, hv, D, D, generator=g)).cuda() for _ in range(2))

    heads = lambda t, h: t.double().view(b, s, h, -1).permute(0, 2, 1, 3).clone().requires_grad_(True)
    q6, k6, v6, be6, al6 = heads(q, hqk), heads(k, hqk), heads(v, hv), heads(be, hv), heads(al, hv)
    s6 = s0.double().requires_grad_(True)
    qr, kr, st, outs = q6.repeat_interleave(hv // hqk, 1), k6.repeat_interleave(hv // hqk, 1), s6, []
    for t in range(s):
        st = st * al6[:, :, t, :, None]
        st = st + (be6[:, :, t] * (v6[:, :, t] - (st * kr[:, :, t, None, :]).sum(-1)))[..., None] * kr[:, :, t, None, :]
        outs.append((st * qr[:, :, t, None, :]).sum(-1) / D**0.5)
    o6 = torch.stack(outs, 2)
    ((o6 * go.double().view(b, s, hv, D).permute(0, 2, 1, 3)).sum() + (st * gs.double()).sum()).backward()
    rows = lambda t: t.detach().permute(0, 2, 1, 3).reshape(b * s, -1)
    want = [rows(o6), rows(q6.grad), rows(k6.grad), rows(v6.grad), st.detach(), rows(be6.grad), rows(al6.grad), s6.grad]
    dist = []
    for chunked in (False, None):
        o, ck, fin = Q.gated_delta_rule_fwd(q, k, v, be, al, b, s, hqk, hv, D, D, state=s0.clone(), chunked=chunked)
        dv = torch.empty_like(v)
        dq, dk, dbe, dal, d0 = Q.gated_delta_rule_bwd(q, k, v, be, al, ck, go, dv, b, s, hqk, hv, D, D, d_final=gs, want_d_initial=True)
        dist.append([rel_l2(x, w) for x, w in zip((o, dq, dk, dv, fin, dbe, dal, d0), want)])
    for i, (one, two) in enumerate(zip(*dist)):
        if i == 7 and decay == "zero":  # behind a decay of zero the first state's gradient is zero itself (here 1e-30 of what it was)
            continue
        assert two < (1.01 * one if i < 4 else 1e-6), (i, one, two)


@pytest.mark.parametrize("what", ["key", "value", "query", "decay", "state"])
def test_chunked_gated_delta_rule_keeps_what_is_not_finite_to_the_rows_behind_it(what):
    """A NaN or an infinity in one token's operands (or the carried state) reaches the outputs that it reaches token by token -- later rows, for a value its own column, for a query its
    own row -- and no row before it in the same chunk; the finite outputs are the same (bf16 rounding flips, as above)."""
    from llm_quest_amd import kernels_q35 as Q

    g = torch.Generator().manual_seed(21)
    D, s, hv, at = 128, 200, 2, 100
    q, k = (torch.nn.functional.normalize(torch.randn(s, hv, D, generator=g), dim=-1).to(BF16).reshape(s, -1).cuda() for _ in range(2))
    v = torch.randn(s, hv * D, generator=g).to(BF16).cuda()
    be, al = torch.sigmoid(torch.randn(s, hv, generator=g)).cuda(), (0.5 + 0.5 * torch.rand(s, hv, generator=g)).cuda()
    s0 = torch.randn(1, hv, D, D, generator=g).cuda()
    if what == "key":
        k[at, 5] = float("nan")
    elif what == "value":
        v[at, 7], v[at + 3, 130] = float("inf"), float("nan")
    elif what == "query":
        q[at, 9] = float("inf")
    elif what == "decay":
        al[at, 1] = float("nan")
    else:
        s0[0, 1, 40, 3] = float("inf")
    out = []
    for chunked in (False, None):
        o, _, fin = Q.gated_delta_rule_fwd(q, k, v, be, al, 1, s, hv, hv, D, D, keep=False, state=s0.clone(), chunked=chunked)
        out.append((o.float(), fin))
    for one, two in zip(*out):
        fine = torch.isfinite(one)
        assert torch.equal(fine, torch.isfinite(two)) and rel_l2(two[fine], one[fine]) < 1e-3
    assert not bool(torch.isfinite(out[1][0]).all()) and bool(torch.isfinite(out[1][0][: (0 if what == "state" else at)]).all())


@pytest.mark.parametrize("what", ["state kept", "state dropped", "not finite"])
def test_chunked_gated_delta_rule_without_a_backward_goes_through_long_sequences_in_spans(what):
    """A forward that keeps nothing has a scratch that does not grow with the sequence (here 18 chunks of 320 heads in spans of ten, 272 MiB for any length)
    and the bits of the forward in one piece."""
    from llm_quest_amd import _lib as L
    from llm_quest_amd import kernels_q35 as Q

    lib, b, hv, s, D = L.load(), 5, 64, 1100, 128
    assert lib.mi355_gdr_chunked_scratch_bytes(b, s, hv) == lib.mi355_gdr_chunked_scratch_bytes(b, 10 * s, hv) < 272 << 20
    assert lib.mi355_gdr_chunked_scratch_bytes(1, s, 16) < 64 << 20
    g = torch.Generator(device="cuda").manual_seed(9)
    r = lambda *z: torch.randn(*z, generator=g, device="cuda")
    q, k = (torch.nn.functional.normalize(r(b * s, 2, D), dim=-1).to(BF16).reshape(b * s, -1) for _ in range(2))
    v, be, al = r(b * s, hv * D).to(BF16), torch.sigmoid(r(b * s, hv)), torch.exp(-torch.exp(r(b * s, hv) - 3.0))
    if what == "not finite":
        v[2 * s + 700, 3] = float("nan")  # (the third sequence, second span)
    s0 = r(b, hv, D, D)
    o, _, fin = Q.gated_delta_rule_fwd(q, k, v, be, al, b, s, 2, hv, D, D, state=s0.clone(), chunked=None)
    bits = lambda t: t.view(torch.int16 if t.dtype == BF16 else torch.int32)
    if what == "state dropped":
        zero, _, _ = Q.gated_delta_rule_fwd(q, k, v, be, al, b, s, 2, hv, D, D, chunked=None)
        o2, _, none = Q.gated_delta_rule_fwd(q, k, v, be, al, b, s, 2, hv, D, D, keep=False, chunked=None)
        assert none is None and torch.equal(bits(o2), bits(zero))
    else:
        o2, _, fin2 = Q.gated_delta_rule_fwd(q, k, v, be, al, b, s, 2, hv, D, D, keep=False, state=s0.clone(), chunked=None)
        fine = torch.isfinite(o.float())
        assert torch.equal(bits(fin2), bits(fin)) or what == "not finite"
        assert torch.equal(fine, torch.isfinite(o2.float())) and torch.equal(torch.isfinite(fin), torch.isfinite(fin2)) and torch.isfinite(fin).any()
        if what == "state kept":
            assert torch.equal(bits(o2), bits(o))
        else:  # (the NaN's column range goes token by token in both, the finite columns of it too)
            assert not bool(fine.all()) and rel_l2(o2.float()[fine], o.float()[fine]) < 1e-3


def test_chunked_gated_delta_rule_refuses_what_it_cannot_read():
    from llm_quest_amd import _lib as L
    from llm_quest_amd import kernels_q35 as Q

    t = torch.zeros(64 * 130, dtype=BF16, device="cuda")
    assert not Q.gdr_chunked(t.view(64, 130)[:, :128], 64, 128, 128) and not Q.gdr_chunked(t[1:].view(-1)[: 64 * 128].view(64, 128), 64, 128, 128)
    assert not Q.gdr_chunked(torch.zeros(63, 128, dtype=BF16, device="cuda"), 63, 128, 128) and not Q.gdr_chunked(torch.zeros(64, 16, dtype=BF16, device="cuda"), 64, 16, 16)
    x, f = torch.zeros(64, 128, dtype=BF16, device="cuda"), torch.zeros(64, 1, device="cuda")
    L.require_gpu(x)
    with pytest.raises(RuntimeError, match="too small"):
        L.call("mi355_gdr_chunked_fwd", 1, 64, 1, 1, L.ptr(x), L.ptr(x), L.ptr(x), 128, L.ptr(f), L.ptr(f), L.ptr(x), L.ptr(f), 16, 0, None, None)


@pytest.mark.parametrize("B,S,C", [(2, 701, 3000), (3, 1, 1398104), (1, 700, 6000)])
def test_causal_conv_of_two_tokens_a_thread(B, S, C):
    """From half a million threads a thread takes two tokens: the same bits as each sequence's channels by themselves, an odd last token, one token alone."""
    from llm_quest_amd import kernels_q35 as Q

    assert B * S * (C // 8) >= 1 << 19
    g = torch.Generator(device="cuda").manual_seed(S)
    x, w = torch.randn(B * S, C + 8, generator=g, device="cuda").to(torch.bfloat16)[:, :C], torch.randn(C, 1, 4, generator=g, device="cuda").to(torch.bfloat16)
    y = Q.causal_conv_silu_fwd(x, w, B, S)
    for b in range(B):
        for c in range(0, C, C // 8 // 3 * 8):
            part = slice(c, min(C, c + C // 8 // 3 * 8))
            assert torch.equal(y[b * S : (b + 1) * S, part], Q.causal_conv_silu_fwd(x[b * S : (b + 1) * S, part], w[part].contiguous(), 1, S))
