"""mi355_attn_generic_fwd / _bwd where their tiles end: query and key tiles of 32, four (head, query tile) pairs to a workgroup, two streams of pairs in the key-major pass."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


@pytest.mark.parametrize("B,S,Hq,Hkv,D,masked", [
    (1, 1, 1, 1, 256, False), (2, 31, 3, 3, 256, False), (1, 32, 4, 1, 256, False), (3, 33, 8, 2, 256, False), (1, 97, 5, 1, 256, True), (2, 160, 8, 2, 256, False),
    (1, 333, 8, 2, 256, False), (2, 65, 4, 4, 256, True), (2, 129, 6, 2, 128, False), (1, 64, 3, 1, 64, True), (2, 95, 2, 2, 32, False)])
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
