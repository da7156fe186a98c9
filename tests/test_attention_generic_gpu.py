"""mi355_attn_generic_fwd / _bwd where their tiles end: query and key tiles of 32, four (head, query tile) pairs to a workgroup, two streams of pairs in the key-major pass."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


@pytest.mark.parametrize("B,S,Hq,Hkv,D,masked", [
    (1, 1, 1, 1, 256, False), (2, 31, 3, 3, 256, False), (1, 32, 4, 1, 256, False), (3, 33, 8, 2, 256, False), (1, 97, 5, 1, 256, True), (2, 160, 8, 2, 256, False),
    (1, 333, 8, 2, 256, False), (2, 65, 4, 4, 256, True), (2, 129, 6, 2, 128, False), (1, 64, 3, 1, 64, True), (2, 95, 2, 2, 32, False),
    # two and four (head, query tile) pairs to a workgroup in the forward pass: from 257 pairs, and from 513 or at small heads
    (4, 130, 16, 2, 256, False), (5, 101, 9, 3, 128, True), (20, 97, 8, 2, 256, False), (21, 70, 6, 2, 128, True), (6, 97, 12, 12, 64, False), (9, 65, 10, 2, 32, True)])
def test_edges_of_tiles_against_64_bits(B, S, Hq, Hkv, D, masked):
    from llm_quest_amd import kernels_q35 as Q

    g = torch.Generator(device="cuda").manual_seed(S * 7 + D)
    rows = torch.randn(B * S, (Hq + 2 * Hkv) * D + 8, generator=g, device="cuda").to(BF16)  # operands inside wider rows
    q, k, v = rows[:, : Hq * D], rows[:, Hq * D : (Hq + Hkv) * D], rows[:, (Hq + Hkv) * D : (Hq + 2 * Hkv) * D]
    do = torch.randn(B * S, Hq * D, generator=g, device="cuda").to(BF16)
    km = None
    allow = torch.ones(S, S, dtype=torch.bool, device="cuda").tril().view(1, 1, S, S)
    if masked:
        km = torch.ones(B, S, dtype=torch.uint8, device="cuda")
        km[0, S - 3 :], km[-1, S // 2] = 0, 0
        allow = allow | (km == 0).view(B, 1, 1, S)
    o, lse = Q.attn_generic_fwd(q, k, v, B, S, Hq, Hkv, D, key_mask=km)
    grads = torch.full_like(rows, 7.0)
    dq, dk, dv = grads[:, : Hq * D], grads[:, Hq * D : (Hq + Hkv) * D], grads[:, (Hq + Hkv) * D : (Hq + 2 * Hkv) * D]
    Q.attn_generic_bwd(q, k, v, o, do, lse, B, S, Hq, Hkv, D, dq, dk, dv, key_mask=km)
    heads = lambda x, H: x.reshape(B, S, H, D).transpose(1, 2).double().contiguous()
    qf, kf, vf = (heads(x, H).requires_grad_(True) for x, H in ((q, Hq), (k, Hkv), (v, Hkv)))
    scores = (qf @ kf.repeat_interleave(Hq // Hkv, 1).mT.contiguous()) * D**-0.5
    ref = torch.softmax(scores.masked_fill(~allow, float("-inf")), -1) @ vf.repeat_interleave(Hq // Hkv, 1)
    ref.backward(heads(do, Hq))
    ref_lse = torch.logsumexp(scores.masked_fill(~allow, float("-inf")), -1)
    # a bf16 rounding is 2^-9 / sqrt(3) = 1.1e-3 of a value in the mean; the forward rounds the weights and the result (1.6e-3 together), the gradients the weights or dS and the
    # result, with delta from a rounded O (dS is a difference of like terms: twice a rounding); the bounds leave a factor of two
    assert float((lse.double().view(B, Hq, S) - ref_lse).detach().abs().max()) < 2e-5
    for name, x, r, H, tol in (("o", o, ref, Hq, 3.5e-3), ("dq", dq, qf.grad, Hq, 6e-3), ("dk", dk, kf.grad, Hkv, 6e-3), ("dv", dv, vf.grad, Hkv, 3.5e-3)):
        err = float((heads(x, H) - r).detach().norm())
        assert err < tol * float(r.detach().norm()) + 1e-3 * (S == 1), (name, err)  # (one key: dQ and dK are zero but for rounding)
    assert bool((grads[:, (Hq + 2 * Hkv) * D :] == 7.0).all())  # nothing beside the gradients was written
    o2, _ = Q.attn_generic_fwd(q, k, v, B, S, Hq, Hkv, D, key_mask=km)
    assert torch.equal(o, o2)


@pytest.mark.parametrize("entry", ["generic", "generic_dropout", "causal_dropout"])
@pytest.mark.parametrize("S,Hq,Hkv,D", [(160, 1, 1, 256), (161, 3, 1, 128), (127, 2, 2, 64), (97, 6, 2, 256), (130, 1, 1, 32)])
def test_a_token_that_is_not_finite_stays_where_it_is_seen(entry, S, Hq, Hkv, D):
    """Without padding a token is seen by itself and later ones: in whole tiles of 32 before it outputs and query gradients keep their bits, in tiles behind a bad query those of the keys
    and values do.  Groups of one, two and three query heads: the four waves of a query-major workgroup stand at different query tiles."""
    from llm_quest_amd import kernels as K, kernels_q35 as Q

    B, bad = 2, S - 20
    g = torch.Generator().manual_seed(S + D)
    q, k, v, do = (torch.randn(B * S, H * D, generator=g).to(BF16).cuda() for H in (Hq, Hkv, Hkv, Hq))

    def run(q, k, v, do):
        grads = [torch.empty_like(t) for t in (q, k, v)]
        if entry == "generic":
            o, lse = Q.attn_generic_fwd(q, k, v, B, S, Hq, Hkv, D)
            Q.attn_generic_bwd(q, k, v, o, do, lse, B, S, Hq, Hkv, D, *grads)
        elif entry == "generic_dropout":
            o, lse = K.attn_generic_dropout_fwd(q, k, v, B, S, Hq, Hkv, D, 0.2, 3, 5)
            K.attn_generic_dropout_bwd(q, k, v, o, do, lse, B, S, Hq, Hkv, D, *grads, 0.2, 3, 5)
        else:
            o, lse = K.attn_dropout_fwd(q, k, v, B, S, Hq, Hkv, D, 0.2, 3, 5, causal=True)
            K.attn_dropout_bwd(q, k, v, o, do, lse, B, S, Hq, Hkv, D, *grads, 0.2, 3, 5, causal=True)
        return [t.view(B, S, -1) for t in (o, *grads)]

    o, dq, dk, dv = run(q, k, v, do)
    before, behind = slice(0, bad // 32 * 32), slice((bad // 32 + 1) * 32, S)
    for value in (float("nan"), float("inf")):
        for which in (1, 2):  # a key, a value
            rows = [q, k, v, do]
            rows[which] = rows[which].clone()
            rows[which].view(B, S, -1)[:, bad] = value
            o1, dq1, _, _ = run(*rows)
            assert torch.equal(o1[:, before], o[:, before]) and torch.equal(dq1[:, before], dq[:, before])
        for which in (0, 3):  # a query, an output gradient
            rows = [q, k, v, do]
            rows[which] = rows[which].clone()
            rows[which].view(B, S, -1)[:, bad] = value
            o1, dq1, dk1, dv1 = run(*rows)
            assert torch.equal(o1[:, before], o[:, before]) and torch.equal(dq1[:, before], dq[:, before])
            assert torch.equal(dk1[:, behind], dk[:, behind]) and torch.equal(dv1[:, behind], dv[:, behind])


@pytest.mark.parametrize("S,Hq,Hkv,D,causal", [(33, 1, 1, 256, True), (97, 4, 2, 256, False), (70, 3, 1, 128, True), (197, 2, 2, 64, False), (5, 2, 1, 32, False)])
def test_the_backward_draws_the_forwards_mask(S, Hq, Hkv, D, causal):
    """dO . O and dV . V are one sum over the kept weights, sum_ij w_ij dO_i . V_j, in every head group: level to the roundings of w, O and dV to bf16 (2^-9 of each, of no fixed sign: 16 times
    that of the terms' 2-norm).  A mask that differs would leave about half that norm."""
    from llm_quest_amd import kernels as K

    B, p = 2, 0.3
    g = torch.Generator().manual_seed(S * D)
    q, k, v, do = (torch.randn(B * S, H * D, generator=g).to(BF16).cuda() for H in (Hq, Hkv, Hkv, Hq))
    grads = [torch.empty_like(t) for t in (q, k, v)]
    o, lse = K.attn_dropout_fwd(q, k, v, B, S, Hq, Hkv, D, p, 11, 13, causal=causal)
    K.attn_dropout_bwd(q, k, v, o, do, lse, B, S, Hq, Hkv, D, *grads, p, 11, 13, causal=causal)
    heads = lambda t, H: t.double().view(B, S, H, D).transpose(1, 2)
    per_group = lambda t: t.reshape(B, Hkv, -1).sum(-1)
    left, right = per_group(heads(o, Hq) * heads(do, Hq)), per_group(heads(v, Hkv) * heads(grads[2], Hkv))
    qd, kd, vd = heads(q, Hq), heads(k, Hkv).repeat_interleave(Hq // Hkv, 1), heads(v, Hkv).repeat_interleave(Hq // Hkv, 1)
    scores = (qd @ kd.mT.contiguous()) * D**-0.5
    if causal:
        scores = scores.masked_fill(torch.ones(S, S, dtype=torch.bool, device="cuda").triu(1), float("-inf"))
    terms = torch.softmax(scores, -1) / (1 - p) * (heads(do, Hq) @ vd.mT.contiguous())
    assert bool(((left - right).abs() <= 16 * 2**-9 * per_group(terms**2).sqrt()).all())
