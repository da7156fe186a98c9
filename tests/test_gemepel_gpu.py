"""GPU tests of the Gemepel serving path against the plain oracle (oracle/gemepel.py): each mechanism's kernel alone, then the model through the
registry, the slot cache and the ragged-batch scheduler -- whole prompts, token-by-token decoding, portions, unequal batches, reused slots, far keys,
odd sizes, greedy generation.  fp32 mode is held to fp32 rounding; bf16 mode to a few bf16 roundings of the logits' scale."""

import json
import math

import pytest
import torch

from oracle import gemepel as G
from tests import gemepel_util as U

pytestmark = pytest.mark.gpu
DEV = "cuda"
F32, BF16, I32 = torch.float32, torch.bfloat16, torch.int32


def dev_i32(x):
    return torch.tensor(x, dtype=I32).to(DEV)


def rel(a, b):
    a, b = a.detach().float().cpu(), b.detach().float().cpu()
    return float((a - b).norm() / (b.norm() + 1e-30))


def row_err(got, want, quantile=None):
    """Per row: rms of the difference (mean removed) over the rms of the wanted rows; the worst row, or a quantile of the rows.

    bf16 runs of whole models are judged on the median row: with random weights and a dozen experts a good part of the tokens has two choice scores
    within a bf16 rounding of the residual stream, and the other expert is then a legitimate choice that moves that token's row.  The fp32 runs, and
    the bf16 runs of every kernel alone, are judged on every row."""
    got, want = got.detach().float().cpu(), want.detach().float().cpu()
    d = got - want
    d = d - d.mean(-1, keepdim=True)
    e = d.pow(2).mean(-1).sqrt() / want.pow(2).mean().sqrt()
    return e.max().item() if quantile is None else torch.quantile(e, quantile).item()


def model_err(got, want, dt):
    return row_err(got, want, None if dt == "float32" else 0.5)


TOL = {"float32": 2e-5, "bfloat16": 6e-2}


# ------------------------------------------------------------------------------------------------------------------- models through the registry
@pytest.fixture(scope="module")
def checkpoint(tmp_path_factory):
    cfg = U.make_config(U.default_layers())
    w = U.make_weights(cfg, 11)
    return U.save(str(tmp_path_factory.mktemp("gemepel")), cfg, w), cfg, w


@pytest.fixture(scope="module")
def models(checkpoint):
    from llm_quest_amd import registry

    folder, cfg, w = checkpoint
    return {dt: registry.load_model(folder, dt, DEV) for dt in ("float32", "bfloat16")}, cfg, w


def tokens(n, vocab, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randint(0, vocab, (n,), generator=g).tolist()


_oracle_cache = {}


def oracle(cfg, w, toks, layers=False):
    key = (id(w), tuple(toks), layers)
    if key not in _oracle_cache:
        _oracle_cache[key] = G.forward(toks, w, cfg, torch.float32, return_layers=layers)
    return _oracle_cache[key]


def batch_of(model, **kw):
    from llm_quest_amd.generate import RaggedBatch

    return RaggedBatch(model, **kw)


@pytest.mark.parametrize("dt", ["float32", "bfloat16"])
def test_whole_prompt_every_layer(models, dt):
    ms, cfg, w = models
    toks = tokens(70, cfg["vocab"], 1)
    want, layers = oracle(cfg, w, toks, layers=True)
    b = batch_of(ms[dt])
    got, got_layers = b.step([("a", toks)], [list(range(len(toks)))], return_layers=True)
    for i, l in enumerate(got_layers):
        assert model_err(l, layers[i], dt) < (2e-5 if dt == "float32" else 8e-2), f"residual stream after layer {i}"
    assert model_err(got, want, dt) < TOL[dt]


@pytest.mark.parametrize("dt", ["float32", "bfloat16"])
def test_token_by_token_from_the_first_token(models, dt):
    """Every token alone: the first one starts the sequence (bigram row of a sequence start, empty state), all others run the continuation path."""
    ms, cfg, w = models
    toks = tokens(45, cfg["vocab"], 2)
    want = oracle(cfg, w, toks)
    b = batch_of(ms[dt])
    got = torch.cat([b.step([("a", [t])]) for t in toks])
    assert model_err(got, want, dt) < TOL[dt]


@pytest.mark.parametrize("dt", ["float32", "bfloat16"])
def test_portions_of_several_sizes(models, dt):
    ms, cfg, w = models
    toks = tokens(90, cfg["vocab"], 3)
    want = oracle(cfg, w, toks)
    b = batch_of(ms[dt])
    got, at = [], 0
    for n in [7, 2, 2, 33, 1, 9, 2, 34]:
        got.append(b.step([("a", toks[at : at + n])], [list(range(n))]))
        at += n
    assert at == len(toks)
    assert model_err(torch.cat(got), want, dt) < TOL[dt]


@pytest.mark.parametrize("dt", ["float32", "bfloat16"])
def test_unequal_batch_equals_each_request_alone(models, dt):
    ms, cfg, w = models
    lens, tail = [3, 41, 17, 66], 9
    seqs = [tokens(n + tail, cfg["vocab"], 10 + i) for i, n in enumerate(lens)]
    alone = []
    for s in seqs:
        b = batch_of(ms[dt])
        alone.append(b.step([("x", s)], [list(range(len(s)))]))
    b = batch_of(ms[dt], slots=2)  # fewer slots than sequences: the cache grows
    got = [[] for _ in seqs]
    out = b.step([(i, s[: lens[i]]) for i, s in enumerate(seqs)], [list(range(n)) for n in lens])
    at = 0
    for i, n in enumerate(lens):
        got[i].append(out[at : at + n])
        at += n
    live = list(range(len(seqs)))
    for k in range(tail):
        if k == 4:  # two requests leave early; the others go on
            for i in (0, 2):
                b.finish(i)
                live.remove(i)
        out = b.step([(i, [seqs[i][lens[i] + k]]) for i in live])
        for j, i in enumerate(live):
            got[i].append(out[j : j + 1])
    for i, s in enumerate(seqs):
        g = torch.cat(got[i])
        ref = alone[i][: g.shape[0]]
        assert model_err(g, ref, dt) < (1e-5 if dt == "float32" else 3e-2), f"request {i} in the batch differs from the request alone"
        assert model_err(g, oracle(cfg, w, s)[: g.shape[0]], dt) < TOL[dt]


def test_freed_slots_are_reused_without_leftovers(models):
    """A long sequence leaves rows and state behind; the next, shorter one takes its slot and must not see any of it.  The cache starts small, so the
    rows also grow while a sequence is alive."""
    ms, cfg, w = models
    b = batch_of(ms["float32"], slots=1)
    b.cache.initial_chunk_size, b.cache.chunk_size = 4, 8
    long_, short = tokens(60, cfg["vocab"], 20), tokens(21, cfg["vocab"], 21)
    b.step([("long", long_[:50])])
    for t in long_[50:]:
        b.step([("long", [t])])
    b.finish("long")
    got = [b.step([("short", short[:12])], [list(range(12))])] + [b.step([("short", [t])]) for t in short[12:]]
    assert b.cache.reuses >= 1 and b.cache.slots == 1
    assert row_err(torch.cat(got), oracle(cfg, w, short)) < TOL["float32"]


def test_long_decoding(models):
    ms, cfg, w = models
    toks = tokens(260, cfg["vocab"], 30)
    b = batch_of(ms["float32"])
    b.step([("a", toks[:5])])
    got = torch.cat([b.step([("a", [t])]) for t in toks[5:]])
    assert row_err(got, oracle(cfg, w, toks)[5:]) < TOL["float32"]


@pytest.mark.parametrize("dt", ["float32", "bfloat16"])
def test_other_sizes_odd_and_one(tmp_path, dt):
    """Sizes that are no multiples of 8, one head, one expert group, top 1, no bigram table, rotation of only part of the rotated entries."""
    from llm_quest_amd import registry

    layers = [(U.latent(heads=1, dim=20, rot_dim=6, vdim=36, q_rank=28, kv_rank=44, rot_dims=4), U.moe(experts=5, top=1, groups=1, keep=1, ff=18)),
              (U.gla(heads=1, dim=10, vdim=70, tau=1.0), U.moe(experts=4, top=4, groups=2, keep=2, ff=30)),
              (U.latent(heads=7, dim=12, rot_dim=6, vdim=20, q_rank=36, kv_rank=44, kv_from=0, rot_dims=4), None),
              (U.gla(heads=4, dim=36, vdim=12, tau=20.0), U.moe(experts=70, top=6, groups=7, keep=3, ff=10))]
    cfg = U.make_config(layers, width=100, vocab=77, eps=1e-6, alpha=1.0, embed_scale=1.0, bigram=None)
    w = U.make_weights(cfg, 5, decay_rank=5)
    model = registry.load_model(U.save(str(tmp_path), cfg, w), dt, DEV)
    toks = tokens(40, cfg["vocab"], 6)
    want = G.forward(toks, w, cfg, torch.float32)
    b = batch_of(model)
    got = [b.step([("a", toks[:29])], [list(range(29))])] + [b.step([("a", [t])]) for t in toks[29:]]
    assert model_err(torch.cat(got), want, dt) < TOL[dt]


def test_greedy_generation_through_the_entry_point(models):
    from llm_quest_amd.generate import generate_ragged

    ms, cfg, w = models
    prompts = [tokens(n, cfg["vocab"], 40 + n) for n in (4, 19, 9)]
    out = generate_ragged(ms["float32"], prompts, max_gen=10)
    for p, gen in zip(prompts, out):
        assert len(gen) == 10
        seq = list(p)
        for t in gen:
            lg = G.forward(seq, w, cfg, torch.float32)[-1]
            top = torch.topk(lg, 2)
            if int(top.indices[0]) != t:
                assert float(top.values[0] - top.values[1]) < 1e-4, "greedy token differs from the oracle's without a near tie"
                break
            seq.append(t)
    # eos ends a sequence early and the others go on
    first = out[1][2]
    out2 = generate_ragged(ms["float32"], prompts, max_gen=10, eos_ids=[first])
    assert out2[1] == out[1][: out[1].index(first)] and out2[0][: len(out2[0])] == out[0][: len(out2[0])]


# ------------------------------------------------------------------------------------------------------------------- mechanisms alone
def test_embedding_first_token_and_large_hash():
    from llm_quest_amd import kernels_seq as S

    vocab, width, buckets, mp, mc = 60000, 24, 1009, 1000003, 999983  # prev * mul_prev overflows 32 bits
    g = torch.Generator().manual_seed(0)
    table, bigram = torch.randn(vocab, width, generator=g).to(BF16), torch.randn(buckets + 1, width, generator=g).to(BF16)
    tok, prev = [59999, 0, 31337, 59998], [-1, 59999, 0, 59997]
    got = S.embed_hash(dev_i32(tok), dev_i32(prev), table.to(DEV), 0.25, bigram.to(DEV), buckets, mp, mc).cpu()
    for i, (t, p) in enumerate(zip(tok, prev)):
        row = buckets if p < 0 else (p * mp + t * mc) % buckets
        assert torch.equal(got[i], table[t].float() * 0.25 + bigram[row].float())


def test_rotary_and_latent_rows_at_large_positions():
    from llm_quest_amd import kernels_seq as S

    T, H, n, dims, start, base = 9, 3, 22, 10, 8, 500000.0
    g = torch.Generator().manual_seed(1)
    x = torch.randn(T, H * n, generator=g)
    pos = [0, 1, 2, 63, 64, 1000, 4095, 4096, 100000]
    freq = S.rope_frequencies(dims, base, DEV)
    dst = torch.zeros(T, H * n, device=DEV)
    S.rope_heads(x.to(DEV), H, n, n, 0, dst, n, 0, start, dims, freq, dev_i32(pos))
    xv = x.view(T, H, n).clone()
    xv[..., start : start + dims] = G.rotate_pairs(xv[..., start : start + dims].double(), torch.tensor(pos), dims, base).float()
    assert (dst.cpu().view(T, H, n)[:8] - xv[:8]).abs().max() < 2e-3  # angle p * f rounds to fp32: up to p * 2^-24 radians
    assert (dst.cpu().view(T, H, n)[:5] - xv[:5]).abs().max() < 1e-5
    assert (dst.cpu().view(T, H, n) - xv).abs().max() < 5e-2
    rank, rot, rd = 20, 12, 8
    src, wgt = torch.randn(T, rank + rot, generator=g), 1 + 0.1 * torch.randn(rank, generator=g)
    cache = torch.zeros(40, rank + rot, device=DEV)
    rows = [3, 39, 0, 7, 8, 21, 22, 23, 30]
    S.latent_kv_append(src.to(DEV), rank, rot, wgt.to(DEV), 1e-5, dev_i32(pos), dev_i32(rows), S.rope_frequencies(rd, base, DEV), rd, cache)
    want_c = G.rms_unit(src[:, :rank], 1e-5) * wgt
    want_r = G.rotate_pairs(src[:, rank:].double(), torch.tensor(pos), rd, base).float()
    got = cache.cpu()[rows]
    assert (got[:, :rank] - want_c).abs().max() < 1e-5 and (got[:5, rank:] - want_r[:5]).abs().max() < 1e-5 and (got[:, rank:] - want_r).abs().max() < 5e-2
    untouched = sorted(set(range(40)) - set(rows))
    assert float(cache.cpu()[untouched].abs().sum()) == 0.0


def _attention_reference(q, k1, k2, v, past, scale):
    """q [n, H, D1+D2], k1 [L, H, D1], k2 [L, D2], v [L, H, DV]: row i sees keys j <= past + i."""
    n, H, _ = q.shape
    D1 = k1.shape[-1]
    out = torch.zeros(n, H, v.shape[-1], dtype=torch.float64)
    for i in range(n):
        L = past + i + 1
        s = (torch.einsum("hd,jhd->hj", q[i, :, :D1], k1[:L]) + q[i, :, D1:] @ k2[:L].T) * scale
        out[i] = torch.einsum("hj,jhd->hd", torch.softmax(s, -1), v[:L])
    return out


@pytest.mark.parametrize("dt", [F32, BF16])
@pytest.mark.parametrize("far", [0, 1, 63, 64, 65, 127, 128, 300, 383])
def test_attention_finds_one_far_key_among_hundreds(dt, far):
    """One key's score stands out (the last query is a multiple of that key): the output must be that key's value, wherever the key lies -- first rows,
    the borders of the 64-key steps, the very last visible key -- in the per-head form (prompt) and in the shared-key form with a past (decoding)."""
    from llm_quest_amd import kernels_seq as S

    H, D1, D2, DV, L = 3, 24, 8, 40, 384
    g = torch.Generator().manual_seed(far)
    k1, k2, v = torch.randn(L, H, D1, generator=g), torch.randn(L, D2, generator=g), torch.randn(L, H, DV, generator=g)
    k1, k2, v = (t.to(dt).float() for t in (k1, k2, v))  # the kernel sees exactly these values in both dtypes
    q = torch.randn(L, H, D1 + D2, generator=g)
    q[-1] = 3.0 * torch.cat([k1[far], k2[far].expand(H, D2)], -1)
    scale = 0.3
    # prompt form: per-head keys and values of this step, no past
    want = _attention_reference(q.double(), k1.double(), k2.double(), v.double(), 0, scale)
    out = torch.empty(L, H * DV, dtype=dt, device=DEV)
    z = dev_i32([0])
    S.latent_attn(q.view(L, -1).to(DEV), k1.view(L, -1).to(dt).to(DEV), k2.to(dt).to(DEV), v.view(L, -1).to(dt).to(DEV), out, H, 1, D1, D2, DV, D1 + D2, D1, DV, DV,
                  (z, dev_i32([L]), z, z, z, z), L, scale)
    tol = 1e-5 if dt == F32 else 2e-2
    assert rel(out.view(L, H, DV), want) < tol
    assert rel(out.view(L, H, DV)[-1], v[far]) < 0.05, "the far key's value did not come through"
    # shared-key form: one key / value row set for all heads (the cache rows), the last 3 rows are new, the rest is the past; rows start at an offset
    ks, vs = k1[:, 0], k1[:, 0]  # keys are also the values, as with cached latent rows
    qs = torch.randn(3, H, D1 + D2, generator=g)
    qs[-1] = 3.0 * torch.cat([ks[far], k2[far]], -1).expand(H, D1 + D2)
    want = _attention_reference(qs.double(), ks[:, None].expand(L, H, D1).double(), k2.double(), vs[:, None].expand(L, H, D1).double(), L - 3, scale)
    off = 5
    rows = torch.zeros(off + L, D1 + D2)
    rows[off:, :D1], rows[off:, D1:] = ks, k2
    rows = rows.to(dt).to(DEV)
    out = torch.empty(3, H * D1, dtype=dt, device=DEV)
    o5 = dev_i32([off])
    S.latent_attn(qs.view(3, -1).to(DEV), rows, rows[:, D1:], rows, out, H, 4, D1, D2, D1, D1 + D2, 0, 0, D1, (z, dev_i32([3]), dev_i32([L - 3]), o5, o5, o5), 3, scale)
    assert rel(out.view(3, H, D1), want) < tol
    assert rel(out.view(3, H, D1)[-1], ks[far].expand(H, D1)) < 0.05


@pytest.mark.parametrize("far", [0, 255, 256, 1023, 1024, 1499])
def test_attention_with_the_keys_dealt_to_several_workgroups(far):
    """One-token steps over a long cache: each tile's keys are split over workgroups and joined afterwards.  Two sequences of different lengths share the
    step; the far key of the longer one lies in the first, a middle or the last share, and at the shares' borders."""
    from llm_quest_amd import kernels_seq as S

    H, D1, D2, L, L2 = 5, 40, 16, 1500, 333
    g = torch.Generator().manual_seed(far)
    rows = torch.randn(L + L2, D1 + D2, generator=g).to(BF16)
    kf = rows.float()
    qs = torch.randn(2, H, D1 + D2, generator=g)
    qs[0] = 3.0 * kf[far]
    scale = 0.25
    want = []
    for n, (lo, hi) in enumerate(((0, L), (L, L + L2))):
        k = kf[lo:hi]
        want.append(_attention_reference(qs[n : n + 1].double(), k[:, None, :D1].expand(-1, H, -1).double(), k[:, D1:].double(), k[:, None, :D1].expand(-1, H, -1).double(),
                                         hi - lo - 1, scale)[0])
    out = torch.empty(2, H * D1, dtype=BF16, device=DEV)
    dr = rows.to(DEV)
    starts = dev_i32([0, L])
    S.latent_attn(qs.view(2, -1).to(DEV), dr, dr[:, D1:], dr, out, H, 8, D1, D2, D1, D1 + D2, 0, 0, D1, (dev_i32([0, 1]), dev_i32([1, 1]), dev_i32([L - 1, L2 - 1]), starts, starts, starts),
                  1, scale, max_keys=L)
    assert S.attn_key_splits(2, 1, 1, 8, L) > 1
    assert rel(out.view(2, H, D1), torch.stack(want)) < 2e-2
    assert rel(out.view(2, H, D1)[0], kf[far, :D1].expand(H, D1)) < 0.05


@pytest.mark.parametrize("dt", [F32, BF16])
def test_gla_kernel_carries_state_over_cuts_and_keeps_a_far_token(dt):
    from llm_quest_amd import kernels_seq as S

    H, dk, dv, T, tau = 2, 20, 70, 150, 4.0
    g = torch.Generator().manual_seed(3)
    q, k, v = (torch.randn(T, H * n, generator=g).to(dt) for n in (dk, dk, dv))
    z = 6.0 + torch.randn(T, H * dk, generator=g)  # decays close to one: the first token stays visible to the end
    k[0] *= 20.0
    bias = 0.5 * torch.randn(H * dk, generator=g)
    qf, kf, vf = q.float().view(T, H, dk), k.float().view(T, H, dk), v.float().view(T, H, dv)
    a = torch.sigmoid((z + bias).double()).pow(1 / tau).view(T, H, dk)
    S_ = torch.zeros(H, dk, dv, dtype=torch.float64)
    want = torch.zeros(T, H, dv, dtype=torch.float64)
    for t in range(T):
        S_ = a[t].unsqueeze(-1) * S_ + kf[t].double().unsqueeze(-1) * vf[t].double().unsqueeze(-2)
        want[t] = torch.einsum("hkv,hk->hv", S_, qf[t].double() * dk ** -0.5)
    state = torch.zeros(3, H, dk, dv, device=DEV)
    state[0] = state[2] = 99.0  # other slots: must stay as they are
    got, at = [], 0
    for n in [1, 7, 8, 9, 16, 1, 1, 2, 105]:  # cuts around the kernel's groups of 8 tokens
        sl = slice(at, at + n)
        got.append(S.gla(q[sl].to(DEV), k[sl].to(DEV), v[sl].to(DEV), z[sl].to(DEV), bias.to(DEV), 1 / tau, dk ** -0.5, dev_i32([0, n]), dev_i32([1]), state, H, dk, dv))
        at += n
    assert at == T
    assert rel(torch.cat(got).view(T, H, dv), want) < 2e-5
    assert rel(state[1], S_) < 2e-5 and float((state[0] - 99).abs().max()) == 0 and float((state[2] - 99).abs().max()) == 0
    contribution = torch.einsum("hk,hv,hk->hv", (a[1:].prod(0) * kf[0].double()), vf[0].double(), qf[-1].double() * dk ** -0.5)
    assert float(contribution.norm() / want[-1].norm()) > 0.5, "the test's far token does not dominate the last output"


def test_router_matches_the_oracle_also_with_negative_choices_and_many_experts():
    from llm_quest_amd import kernels_seq as S

    for E, top, groups, keep, corr_mean in [(8, 2, 2, 1, 0.0), (12, 3, 4, 2, -2.0), (160, 6, 8, 3, -0.4), (70, 5, 70, 9, 0.1), (6, 6, 1, 1, 0.0), (200, 1, 4, 4, -3.0)]:
        g = torch.Generator().manual_seed(E)
        logits, corr = 2 * torch.randn(37, E, generator=g), corr_mean + 0.3 * torch.randn(E, generator=g)
        r = {"experts": E, "top": top, "groups": {"count": groups, "keep": keep}, "scale": 1.7}
        w = {"x.router": torch.eye(E), "x.correction": corr}
        ids, wt = G.route(logits, w, "x.", r)
        gi, gw = S.moe_route(logits.to(DEV), corr.to(DEV), top, groups, keep, 1.7)
        assert torch.equal(gi.cpu().long(), ids), (E, top, groups, keep)
        assert torch.allclose(gw.cpu(), wt, atol=1e-6)
        offs, perm = S.moe_dispatch(gi.view(-1), E)
        offs, perm = offs.cpu().tolist(), perm.cpu().tolist()
        flat = ids.view(-1).tolist()
        assert offs[0] == 0 and offs[-1] == len(flat) and sorted(perm) == list(range(len(flat)))
        for e in range(E):
            assert all(flat[i] == e for i in perm[offs[e] : offs[e + 1]]) and perm[offs[e] : offs[e + 1]] == sorted(perm[offs[e] : offs[e + 1]])


@pytest.mark.parametrize("dt", [F32, BF16])
def test_strided_and_grouped_products(dt):
    from llm_quest_amd import kernels_seq as S

    g = torch.Generator().manual_seed(4)
    # per-head product with the weight read [in, out] (n fastest) and [out, in]
    T, H, dn, R, extra = 37, 3, 20, 44, 6
    a = torch.randn(T, H * (dn + extra), generator=g).to(dt)
    wk = torch.randn(H * dn, R, generator=g).to(BF16)
    c = torch.zeros(T, H * (R + 2), device=DEV)
    S.bgemm(a.to(DEV), wk.to(DEV), c, T, R, dn, batch=H, lda=a.shape[1], a_bs=dn + extra, sbn=1, sbk=R, b_bs=dn * R, ldc=H * (R + 2), c_bs=R + 2)
    want = torch.einsum("thd,hdr->thr", a.float().view(T, H, dn + extra)[..., :dn], wk.float().view(H, dn, R))
    assert rel(c.view(T, H, R + 2)[..., :R], want) < 1e-5
    wv = torch.randn(H * 28, R, generator=g).to(BF16)
    a2 = torch.randn(T, H * R, generator=g).to(dt)
    c2 = torch.empty(T, H * 28, dtype=dt, device=DEV)
    S.bgemm(a2.to(DEV), wv.to(DEV), c2, T, 28, R, batch=H, lda=H * R, a_bs=R, sbn=R, sbk=1, b_bs=28 * R, ldc=H * 28, c_bs=28)
    assert rel(c2.view(T, H, 28), torch.einsum("thr,hvr->thv", a2.float().view(T, H, R), wv.float().view(H, 28, R))) < (1e-5 if dt == F32 else 4e-3)


@pytest.mark.parametrize("dt", ["float32", "bfloat16"])
def test_mixture_of_experts_alone(dt):
    from llm_quest_amd.common.mixers import GroupedSigmoidMoE

    cfg = U.make_config([(U.gla(), U.moe(experts=10, top=3, groups=5, keep=2, ff=36))], width=88)
    w = U.make_weights(cfg, 8)
    m = GroupedSigmoidMoE(88, 36, 10, 3, 5, 2, 2.5)
    m.w_router.data.copy_(w["l0.mlp.router"])
    m.correction.data.copy_(w["l0.mlp.correction"])
    m.w_up.data.copy_(torch.stack([w[f"l0.mlp.e{e}.up"] for e in range(10)]))
    m.w_down.data.copy_(torch.stack([w[f"l0.mlp.e{e}.down"] for e in range(10)]))
    m = m.to(DEV)
    x = torch.randn(150, 88, generator=torch.Generator().manual_seed(9))
    act = F32 if dt == "float32" else BF16
    h = x.to(act)
    got = m.step(x.to(DEV), h.to(DEV)).view(150, 3, 88).sum(1)
    wf = {k: v.float() for k, v in w.items()}
    ids_x, _ = G.route(x, wf, "l0.mlp.", cfg["layers"][0]["mlp"]["router"])
    want = torch.zeros(150, 88)
    _, wt = G.route(x, wf, "l0.mlp.", cfg["layers"][0]["mlp"]["router"])
    for t in range(150):
        for j in range(3):
            e = int(ids_x[t, j])
            want[t] += wt[t, j] * (wf[f"l0.mlp.e{e}.down"] @ (torch.relu(wf[f"l0.mlp.e{e}.up"] @ h[t].float()) ** 2))
    assert rel(got, want) < (1e-5 if dt == "float32" else 1e-2)


def test_post_sum_layernorm_and_head_norm():
    from llm_quest_amd import kernels_seq as S

    g = torch.Generator().manual_seed(6)
    for width in (72, 100, 256, 1000):
        x, y = 3 + torch.randn(13, width, generator=g), torch.randn(13 * 2, width, generator=g)
        w, b = torch.randn(width, generator=g), torch.randn(width, generator=g)
        out, cast = S.add_layernorm(x.to(DEV), w.to(DEV), b.to(DEV), 1e-5, 3.0, y.to(DEV), 2, BF16)
        want = G.layer_norm((3.0 * x + y.view(13, 2, width).sum(1)).double(), w.double(), b.double(), 1e-5)
        assert (out.cpu() - want).abs().max() < 2e-5 and torch.equal(cast.cpu(), out.cpu().to(BF16))
    o, gate, wn = torch.randn(11, 3 * 70, generator=g), torch.randn(11, 3 * 70, generator=g), torch.randn(70, generator=g)
    got = S.gated_headnorm(o.to(DEV), wn.to(DEV), gate.to(DEV), 3, 70, 1e-5, F32)
    want = (G.rms_unit(o.view(11, 3, 70).double(), 1e-5) * wn.double()).view(11, -1) * torch.nn.functional.silu(gate.double())
    assert (got.cpu() - want).abs().max() < 1e-5


# ----------------------------------------------------------------------------------------------- the fp32 product on split operands
@pytest.mark.parametrize("M,N,K", [(1, 32, 8), (3, 33, 24), (31, 1000, 136), (32, 64, 1024), (33, 200, 264), (128, 96, 2048), (129, 130, 2056), (450, 256, 520), (700, 16640, 72)])
def test_fp32_product_on_split_operands(M, N, K):
    """fp32 rows times bf16 weights: edges of the stream's and both tiles' rows, columns and k runs, strided rows, against fp64 -- per output the error of n fp32 roundings of
    the partial sums, n = the 16-steps (three products each) plus the eight runs -- and a row's bits with and without other rows."""
    from llm_quest_amd import kernels_seq as S

    g = torch.Generator().manual_seed(M + N + K)
    wide = (torch.randn(M, K + 12, generator=g) * torch.exp(3 * torch.randn(M, K + 12, generator=g))).cuda()
    x, w = wide[:, 4 : 4 + K], (torch.randn(N, K, generator=g) / K ** 0.5).to(BF16).cuda()
    got = S.linear(x, w)
    want = x.double() @ w.double().T
    bound = (3 * ((K + 15) // 16) + 8 + 16) * 2.0 ** -23 * (x.double().abs() @ w.double().abs().T)
    assert bool(((got.double() - want).abs() <= bound).all())
    for rows in ([M - 1], list(range(0, M, 3)), list(range(M // 2, M))):
        if rows:
            assert torch.equal(S.linear(x[rows].contiguous(), w), got[rows])
    if M > 2:  # infinities and NaN stay what they are, in their rows alone; the largest numbers do not overflow in the split
        y = x.clone()
        y[0, 0], y[1, K - 1], y[2] = float("inf"), float("nan"), 0.0
        y[2, 0] = 3.4028234e38
        out = S.linear(y, w)
        assert torch.equal(out[0].sign(), w[:, 0].float().sign()) and bool(out[0][w[:, 0] != 0].isinf().all()) and bool(out[1].isnan().all())
        big = 3.4028234663852886e38 * w[:, 0].double()
        assert float((out[2].double() - big).abs().max()) <= 2.0 ** -22 * float(big.abs().max()) and torch.equal(out[3:], got[3:])


@pytest.mark.parametrize("M,N,K", [(3, 200, 272), (200, 130, 96), (1024, 8192, 64)])
def test_fp32_product_with_weights_that_are_not_finite(M, N, K):
    """The fp32 product of the stream, the 64-row and the 128-row tiles with infinite and NaN weights: infinite, NaN and finite results are those of fp64, element by element (finite
    columns to fp32 rounding of K exact products)."""
    from llm_quest_amd import kernels_seq as S

    g = torch.Generator().manual_seed(M)
    x, w = torch.randn(M, K, generator=g), torch.randn(N, K, generator=g).to(BF16)
    x[1, 7] = 0.0  # meets an infinity: NaN
    x[2] = x[2].to(BF16).float()  # a bf16 number's second and third parts are zero
    w[0, 7], w[33, K - 1], w[N - 1, 40] = float("inf"), -float("inf"), float("nan")
    w[65, 3], w[65, 50] = float("inf"), -float("inf")
    out = S.linear(x.to(DEV), w.to(DEV), out_dtype=F32).cpu()
    cols = [0, 1, 33, 34, 64, 65, 66, N - 2, N - 1]
    want = (x.double()[:, None, :] * w[cols].double()[None]).sum(-1)
    got = out[:, cols].double()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf()) and torch.equal(got[want.isinf()], want[want.isinf()])
    fine = want.isfinite()
    assert float((got[fine] - want[fine]).abs().max()) < 2e-5 * K**0.5 and bool(out[:, [c for c in range(N) if c not in (0, 33, 65, N - 1)]].isfinite().all())


@pytest.mark.parametrize("rows,groups", [(300, 16), (257, 20)])
def test_grouped_product_with_m_as_the_rows_of_one_group(rows, groups):
    """``M`` may count the rows of the largest group instead of all: the 256 x 256 tiles' grid is then smaller than the work and its workgroups go round.  bf16 operands, fp32 sums and
    results: 2^-24 a sum of K exact products."""
    from llm_quest_amd import kernels_seq as S

    g = torch.Generator().manual_seed(rows)
    N, K, T = 1024, 256, rows * groups
    x, w = torch.randn(T, K, generator=g).to(BF16).to(DEV), torch.randn(groups, N, K, generator=g).to(BF16).to(DEV)
    offs = torch.arange(0, T + 1, rows, dtype=torch.int32, device=DEV)
    out = [torch.full((T, N), float("nan"), device=DEV) for _ in range(2)]
    for o, m in zip(out, (T, rows)):
        S.bgemm(x, w.view(-1, K), o, m, N, K, batch=groups, sbn=K, b_bs=N * K, grp_offs=offs)
    want = torch.cat([x[i * rows : (i + 1) * rows].double() @ w[i].double().T for i in range(groups)])
    assert float((out[0].double() - want).abs().max()) < K * 2.0 ** -24 * 60 and torch.equal(out[0], out[1])


@pytest.mark.parametrize("T,top,epi", [(5, 2, 1), (70, 3, 0), (90, 2, 4), (400, 2, 4)])
def test_fp32_grouped_product_on_split_operands(T, top, epi):
    """Experts (rows gathered, scaled and scattered; one expert without rows; gated blocks): stream and tile against fp64."""
    from llm_quest_amd import kernels_seq as S

    E, K, ff = 5, 200, 96
    g = torch.Generator().manual_seed(T)
    x = torch.randn(T, K, generator=g).cuda()
    ids = torch.stack([torch.randperm(E - 1, generator=g)[:top] for _ in range(T)])
    offs, perm = S.moe_dispatch(ids.reshape(-1).to(torch.int32).cuda(), E)
    n_out = ff // 2 if epi == 4 else ff
    n = 64 * -(-n_out // 32) if epi == 4 else ff
    w = (torch.randn(E, n, K, generator=g) / K ** 0.5).to(BF16).cuda()
    sc = torch.rand(T * top, generator=g).cuda()
    out = torch.zeros((T * top, n_out), device="cuda")
    S.bgemm(x, w, out, T * top, n, K, batch=E, sbn=K, b_bs=n * K, grp_offs=offs, a_rows=perm, a_div=top, c_rows=perm, row_scale=sc, epi=epi, n_out=n_out if epi == 4 else 0)
    y = torch.einsum("tk,tnk->tn", x.double().repeat_interleave(top, 0), w.double()[ids.reshape(-1).cuda()])
    if epi == 4:
        b = y.view(T * top, -1, 2, 32)
        y = (torch.nn.functional.silu(b[:, :, 0]) * b[:, :, 1]).flatten(1)[:, :n_out]
    elif epi == 1:
        y = torch.relu(y) ** 2
    want = y * sc.double()[:, None]
    assert float((out.double() - want).norm() / want.norm()) < 2e-6  # fp32 sums of 200 products and the epilogue's few roundings


@pytest.mark.parametrize("rows,n,K,epi,out", [([1, 0, 31, 257, 600, 256, 65], 2560, 64, 0, F32), ([300, 5, 513], 5700, 128, 1, BF16), ([0, 700, 33, 129], 4096, 192, 4, BF16),
                                              ([2] * 70 + [90], 250, 64, 2, F32), (None, 2050, 64, 0, BF16)])
def test_bf16_product_on_wide_tiles(rows, n, K, epi, out):
    """256 x 256 tiles: groups of uneven rows (none, one, around 32 / 64 / 128 / 256, more groups than lanes), gathered and scattered rows, columns that are no whole words, gated
    blocks; and a plain batch.  fp32 sums of K exact products: results within a few fp32 roundings, resp. one bf16 rounding, of fp64."""
    from llm_quest_amd import kernels_seq as S

    g = torch.Generator().manual_seed(n + K)
    batch, per = (len(rows), None) if rows else (3, 4100)
    R = sum(rows) if rows else per
    gated = epi in (2, 4)
    n_out, n_rows = (n, 64 * -(-n // 32)) if gated else (n, n)
    x = torch.randn(R if rows else batch * R, K + 8, generator=g).to(BF16).cuda()[:, :K]
    w = (torch.randn(batch, n_rows, K, generator=g) / K ** 0.5).to(BF16).cuda()
    total = x.shape[0]
    c = torch.full((total, n_out + 2), 7.0, dtype=out, device="cuda")
    grp, perm, sc = None, None, None
    if rows:
        offs = [0]
        for r in rows:
            offs.append(offs[-1] + r)
        grp, perm = torch.tensor(offs, dtype=torch.int32, device="cuda"), torch.randperm(R, generator=g).to(torch.int32).cuda()
        sc = torch.rand(R, generator=g).cuda()
    S.bgemm(x, w, c, R, n_rows, K, batch=batch, a_bs=0 if rows else R * x.stride(0), sbn=K, b_bs=n_rows * K, c_bs=0 if rows else R * c.stride(0), grp_offs=grp, a_rows=perm, c_rows=perm,
            row_scale=sc, epi=epi, limit=2.5, n_out=n_out if gated else 0)
    bad = 0.0
    for b in range(batch):
        r = perm[offs[b] : offs[b + 1]].long() if rows else torch.arange(b * R, (b + 1) * R, device="cuda")
        if not r.numel():
            continue
        y = x[r].double() @ w[b].double().T
        if gated:
            v = y.view(len(r), -1, 2, 32)
            gt, up = (v[:, :, i].flatten(1)[:, :n] for i in (0, 1))
            y = gt.clamp(max=2.5) * torch.sigmoid(1.702 * gt.clamp(max=2.5)) * (up.clamp(-2.5, 2.5) + 1) if epi == 2 else torch.nn.functional.silu(gt) * up
        elif epi == 1:
            y = torch.relu(y) ** 2
        y = y * sc[r].double()[:, None] if rows else y
        bad = max(bad, float((c[r, :n_out].double() - y).norm() / y.norm()))
    assert bad < (2e-6 if out == F32 else 2.5e-3)
    assert bool((c[:, n_out:] == 7.0).all())  # nothing beside the columns


@pytest.mark.parametrize("T,E,K,top,groups,keep", [(1, 1, 4, 1, 1, 1), (1, 16, 1024, 2, 4, 2), (4, 64, 1024, 6, 8, 3), (3, 65, 100, 4, 5, 2), (4, 128, 520, 8, 1, 1), (3, 240, 512, 70, 4, 4), (2, 512, 256, 3, 16, 5),
                                                   (8, 8, 1744, 8, 2, 2), (5, 32, 512, 3, 8, 2), (7, 24, 64, 5, 2, 1), (9, 16, 1024, 2, 1, 1), (5, 33, 64, 2, 1, 1), (4, 64, 4096, 2, 1, 1), (4, 16, 102, 2, 2, 1)])
def test_choice_of_few_tokens_in_one_launch(T, E, K, top, groups, keep):
    """One launch against the three it stands for: the same ids, weights and lists bit for bit, in every mode, over rows of any pitch and weights of any alignment; what it does not take goes
    the old way."""
    from llm_quest_amd import _lib as L
    from llm_quest_amd import kernels_seq as S

    g = torch.Generator().manual_seed(T * E + K)
    lds = 4 * (T * (K + E + top) + E + 16)
    assert bool(L.load().mi355_moe_choose_takes(T, E, K, top)) == (T <= (8 if E <= 32 else 4) and K % 4 == 0 and E * K <= 1 << 17 and lds <= 65536)
    x = torch.randn(T, K + 3, generator=g).to(DEV)[:, :K]
    for off in (0, 1):
        w = torch.randn(E * K + off, generator=g).to(torch.bfloat16).to(DEV)[off:].view(E, K)
        corr = torch.randn(E, generator=g).to(DEV)
        x[:, 0] = 0.0 if off else x[:, 0]
        for softmax, c in ((False, corr), (False, None), (True, None), ("chosen", corr)):
            if softmax == "chosen" and groups > 1:
                continue
            got = S.moe_choose(x, w, c, top, groups, keep, 1.7, softmax)
            ids, wts = S.moe_route(S.router_logits(x, w), c, top, groups, keep, 1.7, softmax)
            want = (ids, wts, *S.moe_dispatch(ids.view(-1), E))
            assert all(a.shape == b.shape and torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("E,top,groups,keep", [(4, 2, 1, 1), (65, 5, 5, 2), (130, 9, 10, 3), (300, 66, 1, 1), (512, 4, 128, 3)])
def test_choice_of_experts_among_equals_and_none(E, top, groups, keep):
    """The order of the choice: the larger score first, of equals the lower number; -inf and NaN scores are chosen last, as expert 0 with weight 0 once nothing else is left."""
    from llm_quest_amd import kernels_seq as S

    g = torch.Generator().manual_seed(E)
    z = torch.randint(-2, 3, (6, E), generator=g).float()
    corr = torch.zeros(E)
    corr[1::3] = float("-inf")
    z[1, ::2], z[2], z[3, E // 2 :] = float("nan"), float("nan"), -200.0
    for c in (None, corr):
        ids, wts = (t.cpu() for t in S.moe_route(z.to(DEV), None if c is None else c.to(DEV), top, groups, keep, 1.0))
        s = torch.sigmoid(z)
        for t in range(6):
            score = [(float(s[t, e]) + (0.0 if c is None else float(c[e])), e) for e in range(E)]
            ok = [(v, e) for v, e in score if v > float("-inf")]  # (NaN is not)
            if groups > 1:
                per, gs = E // groups, []
                for n in range(groups):
                    two = sorted((v for v, e in ok if e // per == n), reverse=True)[:2] + [float("-inf")] * 2
                    gs.append((-(two[0] + two[1] if per > 1 else two[0]), n))
                kept = {n for _, n in sorted(gs)[:keep]}
                ok = [(v, e) for v, e in ok if e // per in kept]
            want = [e for _, e in sorted(ok, key=lambda x: (-x[0], x[1]))][:top]
            assert ids[t].tolist() == want + [0] * (top - len(want))
            assert not wts[t, len(want) :].any()


@pytest.mark.parametrize("M,N,K", [(129, 128, 1024), (192, 130, 1032), (193, 1, 1096), (450, 1024, 2048), (300, 260, 1992), (1000, 384, 1024), (130, 512, 4096), (450, 1024, 1016)])
def test_tiles_of_eight_waves(M, N, K):
    """Few tiles of a long sum go to eight waves, which divide its shares: the bits of four (the same rows among enough others to fill the chip) over sums that are no whole number of shares or
    steps, and an infinity's row by FMA as ever."""
    from llm_quest_amd import kernels_seq as S

    g, tn = torch.Generator().manual_seed(M + K), (N + 127) // 128
    many = 24576 // tn
    assert tn * ((M + 63) // 64) <= 256 < tn * ((many + 63) // 64) and tn * ((many + 127) // 128) < 512  # 64-row tiles of eight waves (from K = 1 024 on) and of four
    a, w = torch.randn(many, K, generator=g).to(DEV), (torch.randn(N, K, generator=g) * K**-0.5).to(torch.bfloat16).to(DEV)
    a[1, 3], a[M - 1, K - 1] = float("inf"), float("nan")
    few, all_ = torch.empty(M, N, device=DEV), torch.empty(many, N, device=DEV)
    S.bgemm(a[:M], w, few, M, N, K)
    S.bgemm(a, w, all_, many, N, K)
    assert torch.equal(few.view(torch.int32), all_[:M].view(torch.int32))
    want = a[2 : M - 1].double() @ w.double().mT
    assert float((few[2 : M - 1].double() - want).norm()) < 2**-21 * float(want.norm())  # (sums of K products in eight shares, each product 2^-24)


@pytest.mark.parametrize("lens,N,K", [([0, 70, 1, 0, 64, 130], 256, 1024), ([129], 128, 1032), ([3, 200, 0, 65], 192, 1096), ([64, 64, 64], 128, 2048)])
@pytest.mark.parametrize("epi", [0, 1, 2, 4])
def test_tiles_of_eight_waves_in_groups(lens, N, K, epi):
    """The same of gathered and scattered rows in groups, with the row's factor, squared ReLU and the gated epilogues: the bits of four waves, which take the call once a last group makes it a large one."""
    from llm_quest_amd import kernels_seq as S

    g, tn, T, E = torch.Generator().manual_seed(N + K), (N + 127) // 128, sum(lens), len(lens)
    more = 24576 // tn - T
    assert T > 128 and tn * ((T + 63) // 64 + E // 2) <= 256 < tn * ((T + more + 63) // 64) and tn * ((T + more + 127) // 128) < 512
    a, w = torch.randn(T + more, K, generator=g).to(DEV), (torch.randn(E + 1, N, K, generator=g) * K**-0.5).to(torch.bfloat16).to(DEV)
    offs = torch.tensor([0] + [sum(lens[: i + 1]) for i in range(E)] + [T + more], dtype=torch.int32, device=DEV)
    to, scale = torch.randperm(T, generator=g), torch.rand(T + more, generator=g).to(DEV)
    rows = torch.cat([to, torch.arange(T, T + more)]).to(torch.int32).to(DEV)
    width, outs = N // 2 if epi >= 2 else N, []
    for n, groups in ((T, E), (T + more, E + 1)):
        out = torch.full((n, width + 2), 7.0, device=DEV)
        S.bgemm(a, w, out, n, N, K, batch=groups, sbn=K, b_bs=N * K, grp_offs=offs, a_rows=rows, c_rows=rows, row_scale=scale, epi=epi, limit=2.5, n_out=width if epi >= 2 else 0)
        assert bool((out[:, width:] == 7).all())
        outs.append(out[:T, :width])
    assert torch.equal(outs[0], outs[1]) and not bool((outs[0] == 7).any())
    e = max(range(E), key=lambda i: lens[i])
    r = rows[int(offs[e]) : int(offs[e + 1])].long()
    y = a[r].double() @ w[e].double().mT
    if epi >= 2:
        v = y.view(len(r), -1, 2, 32)
        gt, up = (v[:, :, i].flatten(1) for i in (0, 1))
        y = gt.clamp(max=2.5) * torch.sigmoid(1.702 * gt.clamp(max=2.5)) * (up.clamp(-2.5, 2.5) + 1) if epi == 2 else torch.nn.functional.silu(gt) * up
    y = (torch.relu(y) ** 2 if epi == 1 else y) * scale[r].double()[:, None]
    assert float((outs[0][r].double() - y).norm()) < 2**-19 * float(y.norm())  # (the sum's 2^-21, squared or through a gate, and the epilogue's roundings)


@pytest.mark.parametrize("lens,N,K", [([0, 70, 1, 0, 64, 130], 256, 1024), ([65, 0, 0, 200], 128, 2048), ([3] * 60, 64, 1024), ([400, 0, 500], 192, 512)])
@pytest.mark.parametrize("dt", ["fp32", "bf16"])
def test_groups_of_any_length(lens, N, K, dt):
    """Rows of groups, empty ones among them, whichever index of the grid counts row tiles: each group's product is the one it has alone."""
    from llm_quest_amd import kernels_seq as S

    g = torch.Generator().manual_seed(N + K)
    T, E, dtype = sum(lens), len(lens), torch.float32 if dt == "fp32" else torch.bfloat16
    a, w = torch.randn(T, K, generator=g).to(dtype).to(DEV), (torch.randn(E, N, K, generator=g) * K**-0.5).to(torch.bfloat16).to(DEV)
    offs = torch.tensor([0] + [sum(lens[: i + 1]) for i in range(E)], dtype=torch.int32, device=DEV)
    perm = torch.randperm(T, generator=g).to(torch.int32).to(DEV)
    out = torch.full((T, N), 7.0, device=DEV)
    S.bgemm(a, w, out, T, N, K, batch=E, sbn=K, b_bs=N * K, grp_offs=offs, a_rows=perm, a_div=1, c_rows=perm)
    want = torch.empty(T, N, dtype=torch.float64, device=DEV)
    for e in range(E):
        rows = perm[int(offs[e]) : int(offs[e + 1])].long()
        want[rows] = a[rows].double() @ w[e].double().mT
    assert float((out.double() - want).norm()) < 2**-20 * float(want.norm())


@pytest.mark.parametrize("T,H,D", [(1, 1, 1), (3, 5, 63), (7, 3, 64), (5, 2, 65), (2, 4, 128), (3, 2, 129), (2, 1, 256), (2, 2, 257), (1024, 12, 64), (4097, 3, 128), (1537, 8, 200), (2000, 16, 96),
                                   (2100, 16, 128), (4099, 16, 64), (8193, 16, 128)])
def test_heads_of_a_wave(T, H, D):
    """Kernels whose waves take several heads from some 12 000 on: one head to a wave or many (of rotations two
    from 1 024 tokens of 16 heads on, four from 2 048, eight from 4 096, all from 8 192), the rows' bits are those of the same rows in a short call; sizes around 64 values a lane's word, rotations of every lane's pair."""
    from llm_quest_amd import _lib as L
    from llm_quest_amd import kernels_seq as S

    g = torch.Generator().manual_seed(T + D)
    few = min(T, 5)
    o, gate = torch.randn(T, H * D, generator=g).to(DEV), torch.randn(T, H * D + 3, generator=g).to(torch.bfloat16).to(DEV)[:, 1 : H * D + 1]
    w, freq, pos = torch.randn(D, generator=g).to(DEV), torch.rand(max(D // 2, 1), generator=g).to(DEV), torch.arange(T, dtype=torch.int32, device=DEV)
    big, small = S.gated_headnorm(o, w, gate, H, D, 1e-6, torch.float32), S.gated_headnorm(o[:few].contiguous(), w, gate[:few], H, D, 1e-6, torch.float32)
    assert torch.equal(big[:few], small)
    x, z = o.double().view(T, H, D), gate.double().view(T, H, D)
    want = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-6) * w.double() * z * torch.sigmoid(z)
    assert float((big.double().view(T, H, D) - want).norm()) < 1e-6 * float(want.norm())
    for dims in {0, D // 2, D // 4 * 2, D if D <= 128 else 128}:
        dims -= dims % 2
        for layout in (0, 1):
            outs = []
            for n in (T, few):
                dst = torch.full((n, H * D), 7.0, device=DEV)
                S.rope_heads(o[:n], H, D, D, 0, dst, D, 0, D - dims, dims, freq, pos[:n], layout)
                outs.append(dst)
            assert torch.equal(outs[0][:few], outs[1]) and not bool((outs[0] == 7).all())
            i = torch.arange(dims // 2, device=DEV)
            a, b = (i, i + dims // 2) if layout else (2 * i, 2 * i + 1)
            ang = (pos.float()[:, None, None] * freq[: dims // 2]).double()
            want = x.clone()
            u, v = x[..., D - dims + a], x[..., D - dims + b]
            want[..., D - dims + a], want[..., D - dims + b] = u * ang.cos() - v * ang.sin(), v * ang.cos() + u * ang.sin()
            assert float((outs[0].double().view(T, H, D) - want).norm()) < 1e-6 * float(want.norm())
    if D <= 256:
        q, k, b, a = (torch.randn(T, n, generator=g).to(DEV) for n in (H * D, H * D, H, H))
        A, dt, ws = torch.randn(H, generator=g).to(DEV), torch.randn(H, generator=g).to(DEV), []
        L.require_gpu(q, k)
        for n in (T, few):
            ws.append(torch.empty(n, H, 4, device=DEV))
            L.call("mi355_delta_rule_tokens", n, H, H, D, L.ptr(q), L.ptr(k), L.DT_F32, q.stride(0), k.stride(0), L.ptr(b), L.ptr(a), L.DT_F32, H, H, L.ptr(A), L.ptr(dt), 0.5, L.ptr(ws[-1]))
        assert torch.equal(ws[0][:few], ws[1])
        kd, qd = k.double().view(T, H, D), q.double().view(T, H, D)
        want = torch.stack([torch.exp(-A.double().exp() * torch.nn.functional.softplus(a.double() + dt.double())), torch.sigmoid(b.double()), ((kd * kd).sum(-1) + 1e-6).rsqrt(), 0.5 * ((qd * qd).sum(-1) + 1e-6).rsqrt()], -1)
        assert float((ws[0].double() - want).norm()) < 1e-6 * float(want.norm())
