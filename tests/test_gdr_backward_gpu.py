"""The chunked gated delta rule's backward: last chunks of every kind, value gradients in views of any alignment, tokens that belong to the next sequence."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def _operands(B, S, Hqk, Hv, seed):
    g = torch.Generator().manual_seed(seed)
    unit = lambda x: torch.nn.functional.normalize(x, dim=-1)
    q, k = (unit(torch.randn(B * S, Hqk, 128, generator=g)).reshape(B * S, -1).to(BF16).cuda() for _ in range(2))
    v, do = (torch.randn(B * S, Hv * 128, generator=g).to(BF16).cuda() for _ in range(2))
    return q, k, v, torch.rand(B * S, Hv, generator=g).cuda(), torch.exp(-0.3 * torch.rand(B * S, Hv, generator=g)).cuda(), do


def _backward(q, k, v, beta, alpha, do, dv, B, S, Hqk, Hv):
    from llm_quest_amd import kernels_q35 as K

    _, ck, _ = K.gated_delta_rule_fwd(q, k, v, beta, alpha, B, S, Hqk, Hv, 128, 128, chunked=None)
    assert ck.dim() == 1  # the chunked kernels'
    return K.gated_delta_rule_bwd(q, k, v, beta, alpha, ck, do, dv, B, S, Hqk, Hv, 128, 128)


@pytest.mark.parametrize("S,Hqk,Hv", [(64, 2, 2), (65, 1, 2), (95, 2, 2), (96, 1, 1), (97, 1, 3), (127, 2, 2), (193, 1, 1)])
def test_last_chunks_and_views(S, Hqk, Hv):
    """Gradients against 64 bits (bf16 results: 2^-9 of a value; fp32 ones: chains of 128 products, 2^-24 each), into rows of any alignment with the same bits, and the first sequence's
    untouched by NaNs in the second's tokens."""
    B = 2
    q, k, v, beta, alpha, do = _operands(B, S, Hqk, Hv, S)
    dv = torch.empty_like(v)
    got = (*_backward(q, k, v, beta, alpha, do, dv, B, S, Hqk, Hv), dv)
    for pad, at in ((1, 1), (4, 4), (6, 2)):
        wide = torch.full((B * S, Hv * 128 + pad + at), 7.0, dtype=BF16, device="cuda")
        view = wide[:, at : at + Hv * 128]
        again = (*_backward(q, k, v, beta, alpha, do, view, B, S, Hqk, Hv), view)
        assert all(torch.equal(a, b) for a, b in zip(got, again)) and bool((wide[:, :at] == 7).all()) and bool((wide[:, at + Hv * 128 :] == 7).all())
    rep = Hv // Hqk
    hd = lambda t: t.double().view(B, S, -1, 128)
    leaves = [hd(q), hd(k), hd(v), beta.double().view(B, S, Hv), alpha.double().view(B, S, Hv)]
    leaves = [t.requires_grad_() for t in leaves]
    qd, kd = leaves[0].repeat_interleave(rep, 2), leaves[1].repeat_interleave(rep, 2)
    st, out = torch.zeros(B, Hv, 128, 128, dtype=torch.float64, device="cuda"), []
    for t in range(S):
        st = st * leaves[4][:, t, :, None, None]
        u = leaves[3][:, t, :, None] * (leaves[2][:, t] - (st * kd[:, t, :, None]).sum(-1))
        st = st + u[..., None] * kd[:, t, :, None]
        out.append((st * qd[:, t, :, None]).sum(-1) * 128**-0.5)
    (torch.stack(out, 1) * hd(do)).sum().backward()
    want = [t.grad.reshape(B * S, -1) for t in leaves]
    for a, b, tol in zip((got[0], got[1], got[4], got[2], got[3]), want, (2**-8, 2**-8, 2**-8, 128 * 2**-24, 128 * 2**-24)):
        assert float((a.double() - b).norm()) < tol * float(b.norm())
    for t in (q, k, v, do):
        t[S:] = float("nan")
    lost = (*_backward(q, k, v, beta, alpha, do, dv, B, S, Hqk, Hv), dv)
    assert all(torch.equal(a[:S], b[:S]) for a, b in zip(got[:4], lost)) and bool(torch.isfinite(lost[4][:S].float()).all())


@pytest.mark.parametrize("S", [64, 65, 96, 130])
def test_output_gradients_reach_no_later_token(S):
    """A dO that is not finite reaches the tokens up to its own; of those behind it, its own 32 at most (in which zeros are multiplied)."""
    B, Hqk, Hv = 1, 1, 2
    q, k, v, beta, alpha, do = _operands(B, S, Hqk, Hv, S)
    dv = torch.empty_like(v)
    want = (*_backward(q, k, v, beta, alpha, do, dv, B, S, Hqk, Hv), dv)
    for t in [t for t in (0, 17, 31, 32, 40, 63, 64, 97, 128) if t < S]:
        for x in (float("inf"), float("nan")):
            bad, dv = do.clone(), torch.empty_like(v)
            bad[t, 130] = x
            got = (*_backward(q, k, v, beta, alpha, bad, dv, B, S, Hqk, Hv), dv)
            later = t // 32 * 32 + 32
            assert all(torch.equal(a[later:], b[later:]) for a, b in zip(got, want)) and not bool(torch.isfinite(got[0][t].float()).all())


@pytest.mark.parametrize("S,decay,size", [(64, 0.3, 1.0), (65, 8.0, 1e30), (96, 0.0, 1e-30), (127, 0.01, 1.0), (129, 8.0, 1.0), (192, 0.001, 1e30), (321, 0.3, 1e-3)])
def test_state_from_a_state(S, decay, size):
    """The final state and the outputs of chunks that start from a state, against 64 bits, over whole and last chunks, decays from none to strong, and sizes where the parts of a split number come
    near either end of fp32.  The state is a sum over 64 tokens a chunk of fp32 products, each rounding 2^-24 of it at most, of U that summed 128 the same way; outputs are bf16."""
    from llm_quest_amd import kernels_q35 as K

    B, Hqk, Hv = 2, 1, 2
    q, k, v, beta, _, _ = _operands(B, S, Hqk, Hv, S)
    g = torch.Generator().manual_seed(S + 1)
    v, alpha = (v.float() * size).to(BF16), torch.exp(-decay * torch.rand(B * S, Hv, generator=g)).cuda()
    st = (torch.randn(B, Hv, 128, 128, generator=g) * size).cuda()
    hd = lambda t: t.double().view(B, S, -1, 128)
    qd, kd, vd, bd, ad, want, out = hd(q).repeat_interleave(Hv, 2), hd(k).repeat_interleave(Hv, 2), hd(v), beta.double().view(B, S, Hv), alpha.double().view(B, S, Hv), st.double(), []
    for t in range(S):
        want = want * ad[:, t, :, None, None]
        u = bd[:, t, :, None] * (vd[:, t] - (want * kd[:, t, :, None]).sum(-1))
        want = want + u[..., None] * kd[:, t, :, None]
        out.append((want * qd[:, t, :, None]).sum(-1) * 128**-0.5)
    out = torch.stack(out, 1).reshape(B * S, -1)
    for keep in (True, False):
        o, _, fin = K.gated_delta_rule_fwd(q, k, v, beta, alpha, B, S, Hqk, Hv, 128, 128, keep=keep, want_state=True, state=st.clone(), chunked=True)
        assert float((fin.double() - want).norm()) < 64 * 2**-24 * float(want.norm())
        assert float((o.double() - out).norm()) < 2**-8 * float(out.norm())
