"""One-token steps where their launches change shape: rows requested by the host's bound, splits folded by the output projection, weight streams of eight-row groups and twelve waves."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


@pytest.mark.parametrize("D,cap,length,wp,splits", [(128, 1, 1, 0, 1), (128, 130, 129, 128, 1), (128, 640, 17, 16, 1), (64, 257, 257, 100, 2), (128, 300, 300, 300, 3), (64, 128, 128, -1, 1),
                                                    (128, 700, 560, 559, 5), (128, 5000, 40, 39, 1)])
def test_rows_requested_by_the_bound_are_those_of_the_length(D, cap, length, wp, splits):
    """Whatever lies past the length is not seen (here: NaN), the new token comes from the launch wherever its row is, and a row at the bound that is an old one is read."""
    from llm_quest_amd import kernels as KK
    from llm_quest_amd import ops_decode

    B, Hq, Hkv = 2, 4, 2
    g = torch.Generator().manual_seed(cap + length)
    rnd = lambda *s: torch.randn(*s, generator=g).to(BF16).cuda()
    qkv, qw, kw = rnd(B, (Hq + 2 * Hkv) * D), rnd(D), rnd(D)
    cos, sin = torch.rand(64, D, generator=g).cuda(), torch.rand(64, D, generator=g).cuda()
    pos = torch.tensor([3, 60], dtype=torch.int32, device="cuda")
    at, n = torch.tensor([wp], dtype=torch.int32, device="cuda"), torch.tensor([length], dtype=torch.int32, device="cuda")
    kc, vc = rnd(B, cap, Hkv * D), rnd(B, cap, Hkv * D)
    kc[:, length:], vc[:, length:] = float("nan"), float("nan")
    q, k, _ = KK.qknorm_rope_fwd(qkv, qw, kw, cos, sin, pos, Hq, Hkv, D)
    kr, vr = kc.clone(), vc.clone()
    if 0 <= wp < cap:
        kr[:, wp], vr[:, wp] = k, qkv[:, (Hq + Hkv) * D :]
    want = ops_decode.attn_decode(q, kr, vr, cap, Hq, Hkv, D, len_dev=n, splits=splits)
    got = ops_decode.attn_decode_qkv(qkv, qw, kw, cos, sin, pos, Hq, Hkv, D, kc, vc, at, n, splits=splits)
    assert torch.equal(got, want) and bool(torch.isfinite(got.float()).all())
    assert torch.equal(kc[:, :length], kr[:, :length]) and torch.equal(vc[:, :length], vr[:, :length])
    heads = lambda x, H: x[:, :length].double().unflatten(2, (H, D)).transpose(1, 2)
    s = (q.double().view(B, Hq, 1, D) @ heads(kr, Hkv).repeat_interleave(2, 1).mT.contiguous()) * D**-0.5
    ref = (torch.softmax(s, -1) @ heads(vr, Hkv).repeat_interleave(2, 1).contiguous()).view(B, Hq * D)
    assert float((got.double() - ref).norm()) < 2.3e-3 * float(ref.norm())  # one bf16 rounding of the result: at most 2^-9 of a value


@pytest.mark.parametrize("past,D", [(255, 64), (256, 128), (257, 64), (640, 128), (1400, 64)])
def test_splits_folded_by_the_projection_equal_the_combining_launch(monkeypatch, past, D):
    from llm_quest_amd import ops_decode as OD
    from llm_quest_amd.qwen.qwen3.qwen3_transformer_block import TransformerBlock
    from llm_quest_amd.utils import KVCache

    torch.manual_seed(past)
    Hq, Hkv, d, hidden = 6, 2, 264, 3000
    with torch.device("cuda"):
        blk = TransformerBlock(dict(emb_dim=d, hidden_dim=hidden, n_heads=Hq, num_kv_groups=Hkv, head_dim=D, dtype=BF16), 0)
        for p in blk.parameters():
            torch.nn.init.normal_(p, std=0.1)
    ang = torch.rand(2048, D // 2, device="cuda")
    cos, sin = torch.cat([ang.cos()] * 2, 1).contiguous(), torch.cat([ang.sin()] * 2, 1).contiguous()
    h = torch.randn(1, d, device="cuda").to(BF16)
    rows = [torch.randn(past, Hkv * D, device="cuda").to(BF16) for _ in range(2)]
    step, outs = OD._block_step, []
    for one in (True, False):
        monkeypatch.setattr(OD, "_block_step", step if one else (lambda *a: None))
        c = KVCache(num_layers=1, prompt_len=past, context_len=2048)
        c.append_rows(*rows, 0, 1, past)
        outs.append(OD.block_cached(blk, h, 1, 1, cos, sin, torch.full((1,), past, dtype=torch.int32, device="cuda"), None, c))
    assert torch.equal(*outs)


@pytest.mark.parametrize("M", [2, 5, 8])
@pytest.mark.parametrize("N,K", [(1, 2048), (8, 2056), (9, 3072), (127, 64), (2048, 264), (2049, 2304), (2056, 3080)])
def test_weight_streams_of_every_shape_of_launch(M, N, K):
    from llm_quest_amd import ops_decode

    g = torch.Generator(device="cuda").manual_seed(N + K)
    x, w, r = (torch.randn(*s, generator=g, device="cuda").to(BF16) for s in ((M, K), (N, K), (M, N)))
    ref = x.double() @ w.double().T.contiguous() + r.double()
    got = ops_decode.gemv(x, w, residual=r)
    # fp32 sums of K exact products, then one bf16 rounding: half a step of 2^-8, the sums' own error far below
    assert bool(((got.double() - ref).abs() <= ref.abs() * 2**-8 + K**0.5 * 1e-5).all())


@pytest.mark.parametrize("B,layers,masked,device_side", [(1, 1, False, False), (1, 4, True, False), (3, 5, False, False), (8, 7, True, False), (9, 3, False, False), (2, 6, False, True), (1, 5, True, True)])
def test_layers_behind_one_call_are_the_layers_one_by_one(monkeypatch, B, layers, masked, device_side):
    """Even and odd counts of layers to a call, a cache that grows in the step, a layer in the middle that takes the separate calls; logits and caches the same bits."""
    from llm_quest_amd import ops_decode as OD
    from llm_quest_amd.qwen.qwen3.qwen3_model import Qwen3Model
    from llm_quest_amd.utils import KVCache

    torch.manual_seed(B + layers)
    past = 5
    with torch.device("cuda"):
        m = Qwen3Model(dict(vocab_size=300, emb_dim=64, n_layers=layers, n_heads=4, num_kv_groups=2, hidden_dim=136, head_dim=64, rope_base=10_000, context_length=64, dtype=BF16, tie_embeddings=True,
                            model_type="dense")).eval()
    ids = torch.randint(0, 300, (B, past + 3), device="cuda")
    km = (torch.rand(B, 1024, device="cuda") < 0.7) if masked else None
    operands, outs = OD._layer_operands, []
    for how in ("all", "all but the third", "none"):
        monkeypatch.setattr(OD, "_layer_operands", lambda blk, i, *a: None if how == "none" or (how != "all" and i == 2) else operands(blk, i, *a))
        c = KVCache(num_layers=layers, prompt_len=past, context_len=64)
        with torch.inference_mode():
            seen = [m(ids[:, :past], kv_cache=c, attn_mask=None if km is None else km[:, :past])]
            if device_side:
                c.reserve(past + 3)
            for t in range(3):
                at = lambda v: torch.tensor([v], dtype=torch.int32, device="cuda")
                state = (at(past + t).repeat(B), at(past + t), at(past + t + 1), 1) if device_side else None
                seen.append(OD.qwen3_forward_cached(m, ids[:, past + t : past + t + 1], c, attn_mask=km, dev_state=state))
                if device_side:
                    c.start_pos += 1
        assert c.start_pos == past + 3
        outs.append(seen + [x[:, : past + 3].clone() for x in c.keys_cache + c.values_cache])
    for got in outs[:-1]:
        assert all(torch.equal(a, b) for a, b in zip(got, outs[-1]))
