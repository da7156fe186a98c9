"""fp32 steps of few tokens on ragged batches: products of few fp32 rows, attention of one or two new tokens, gated linear attention by groups of tokens."""
import pytest
import torch

pytestmark = pytest.mark.gpu
F32, BF16 = torch.float32, torch.bfloat16
EPS = 2.0**-24


def i32(x):
    return torch.tensor(x, dtype=torch.int32, device="cuda")


@pytest.mark.parametrize("M,K,N", [(1, 8, 7), (1, 256, 1024), (3, 1000, 1032), (32, 520, 1025), (31, 704, 33 * 32), (7, 2056, 192 * 32 + 8), (2, 1024, 193 * 32), (9, 2560, 40), (12, 2048, 96)])
def test_product_of_few_fp32_rows_has_the_bits_of_many(M, K, N):
    """8, 16 or 32 columns a workgroup, wave runs of no, one, and several stages, rows that fit LDS and rows that just do not (9 x 2560 and 12 x 2048 are on both sides of it): the
    product of the same rows among 129 goes through the tile kernel, whose sums are the same.  Against 64 bits: 3 parts x K products, each sum rounded, and the wave's sums."""
    from llm_quest_amd import kernels_seq as S

    g = torch.Generator().manual_seed(M + K + N)
    x = torch.randn(129, K, generator=g).cuda()
    x[:M] *= torch.logspace(-12, 12, K, base=2.0).cuda()[torch.randperm(K, generator=g).cuda()]
    w = torch.randn(N, K, generator=g).to(BF16).cuda()
    got, many = S.linear(x[:M], w), S.linear(x, w)
    assert torch.equal(got, many[:M])
    bound = (K + 16) * EPS * (x[:M].double().abs() @ w.double().abs().T)
    assert bool(((got.double() - x[:M].double() @ w.double().T).abs() <= bound).all())
    x[0, 0], x[M - 1, K - 1] = float("inf"), float("nan")
    torch.testing.assert_close(S.linear(x[:M], w), S.linear(x, w)[:M], rtol=0, atol=0, equal_nan=True)


@pytest.mark.parametrize("counts,K,N,epi,dt", [([0, 3, 1, 0, 2], 1792, 1024, 0, F32), ([32], 264, 70, 1, F32), ([1, 0, 5], 520, 2 * 64, 4, F32), ([40, 1, 0, 33], 520, 64 * 3, 4, BF16),
                                               ([0, 2, 70], 1000, 100, 1, BF16), ([6] * 20, 264, 40, 0, BF16), ([3, 0, 90], 320, 64, 0, F32)])
def test_experts_of_few_rows(counts, K, N, epi, dt):
    """Streams of the weights of groups with few rows, gathered and scattered; wave runs of no, one and several stages; experts without rows; more rows than one workgroup holds."""
    from llm_quest_amd import kernels_seq as S

    E, R = len(counts), sum(counts)
    g = torch.Generator().manual_seed(R + K)
    x = torch.randn(R, K, generator=g).to(dt).cuda()
    w = (torch.randn(E, N, K, generator=g) / K**0.5).to(BF16).cuda()
    perm = torch.randperm(R, generator=g).to(torch.int32).cuda()
    sc = torch.rand(R, generator=g).cuda()
    offs = i32([0] + torch.tensor(counts).cumsum(0).tolist())
    n_out = N // 2 if epi == 4 else N
    out = torch.full((R, n_out), float("nan"), device="cuda")
    S.bgemm(x, w, out, R, N, K, batch=E, sbn=K, b_bs=N * K, grp_offs=offs, a_rows=perm, c_rows=perm, row_scale=sc, epi=epi, n_out=n_out if epi == 4 else 0)
    for e in range(E):
        r = perm[offs[e] : offs[e + 1]].long()
        y, mag = x[r].double() @ w[e].double().T, x[r].double().abs() @ w[e].double().abs().T
        err = (K + 16) * EPS * mag
        if epi == 4:  # |d silu| < 1.1, |silu(a)| <= |a|; the gate's few roundings
            a, b = y.view(len(r), N // 64, 2, 32).unbind(2)
            ea, eb = err.view(len(r), N // 64, 2, 32).unbind(2)
            y = (torch.nn.functional.silu(a) * b).flatten(1)
            err = (1.1 * ea * b.abs() + eb * a.abs() + 8 * EPS * (a * b).abs()).flatten(1)
        elif epi == 1:
            y, err = torch.relu(y) ** 2, 2 * mag * err
        s = sc[r].double()[:, None]
        assert bool(((out[r].double() - y * s).abs() <= err * s + 4 * EPS * (y * s).abs()).all())


CASES = [dict(), dict(shared=True, D2=8), dict(shared=True, values_are_keys=True, D1=256, D2=64, DV=256, H=8), dict(H=6, rep=3, DV=70), dict(H=8, rep=4, window=37, keep=5), dict(H=4, rep=2, chunk=48),
         dict(H=3, window=20, chunk=64, softcap=3.0), dict(H=5, shared=True, sink=True, slope=True), dict(H=2, sig=True, window=33), dict(H=4, gate=True, softcap=2.0, D1=130, DV=257),
         dict(H=9, shared=True, D1=512, D2=128, DV=512, values_are_keys=True), dict(H=2, D1=100, DV=129, window=1), dict(H=4, rep=4, sink=True, window=16, keep=64)]
# values that are the first features of the keys and come by the keys' row table itself (the served models' call): read once, in every size of the kernel
CASES += [dict(opt, values_are_keys=True, one_table=True) for opt in (dict(shared=True, D1=72, D2=8, DV=48, H=5), dict(shared=True, D1=200, DV=150, H=4, sink=True), dict(shared=True, D1=256, D2=64, DV=256, H=8, window=37),
                                                                      dict(shared=True, D1=512, D2=128, DV=512, H=9), dict(H=6, rep=3, D1=64, DV=64), dict(H=8, rep=4, D1=130, DV=129, sig=True))]


@pytest.mark.parametrize("opt", CASES, ids=lambda o: "-".join(f"{k}{int(v)}" for k, v in o.items()) or "plain")
@pytest.mark.parametrize("dt", [F32, BF16])
def test_attention_of_one_or_two_new_tokens(opt, dt):
    """Sequences of 1, 2 and 3 new tokens after 0 .. 200 keys in one step, every option; the rows of a sequence are bit by bit those it has alone.  Scores are sums of D products and
    a weight's relative error is its score's error; the values' sum over n keys rounds n times: 64 bits within 2^-24 (n + |q||k| scale (D + 4)) of the largest weighted value."""
    from llm_quest_amd import kernels_seq as S

    H, D1, D2, DV = opt.get("H", 2), opt.get("D1", 64), opt.get("D2", 0), opt.get("DV", 48)
    rep, shared, same = opt.get("rep", 1), opt.get("shared", False), opt.get("values_are_keys", False)
    window, keep, chunk, cap = opt.get("window", 0), opt.get("keep", 0), opt.get("chunk", 0), opt.get("softcap", 0.0)
    new, past = [1, 2, 3, 1, 2, 1, 1], [0, 0, 5, 31, 64, 129, 200]
    g = torch.Generator().manual_seed(H * D1 + DV)
    G = 1 if shared else H // rep
    total = [n + p for n, p in zip(new, past)]
    T, R = sum(total), sum(new)
    k1, k2 = torch.randn(T, G * D1, generator=g).to(dt).cuda(), torch.randn(T, max(D2, 1), generator=g).to(dt).cuda()
    v = k1 if same else torch.randn(T, G * DV, generator=g).to(dt).cuda()
    q = (torch.randn(R, H * (D1 + D2), generator=g)).cuda()
    sink, slope, sig = [torch.randn(H, generator=g).cuda() if opt.get(n) else None for n in ("sink", "slope", "sig")]
    slope = slope.abs() * 0.1 if slope is not None else None
    gate = torch.randn(R, H * DV, generator=g).cuda() if opt.get("gate") else None
    scale = (D1 + D2) ** -0.5
    cum = lambda a: [sum(a[:i]) for i in range(len(a))]
    q0, k0 = cum(new), cum(total)

    def run(seqs):
        out = torch.full((R, H * DV), float("nan"), device="cuda")
        pick = lambda a: i32([a[i] for i in seqs])
        table = pick(k0)
        desc = (pick(q0), pick(new), pick(past), table, pick(k0), table if opt.get("one_table") else pick(k0))
        hm = 1
        while hm * 2 <= 8 and (shared or rep % (hm * 2) == 0):
            hm *= 2
        return _fp32_path(S, q, k1, k2 if D2 else None, v, out, H, hm, D1, D2, DV, shared, desc, max(new[i] for i in seqs), scale, 1 if shared else rep, window, keep, cap, sink, chunk, sig, slope, gate)

    got = run(list(range(len(new))))
    for i in range(len(new)):
        rows = slice(q0[i], q0[i] + new[i])
        assert torch.equal(got[rows], run([i])[rows])
        if i >= 2:
            assert torch.equal(got[rows], run([0, i])[rows]) and torch.equal(got[rows], run([i, 2] if i != 2 else [2, 6])[rows])
        n = total[i]
        ks = k1[k0[i] : k0[i] + n].double().view(n, G, D1).expand(n, H, D1) if shared else k1[k0[i] : k0[i] + n].double().view(n, G, D1).repeat_interleave(rep, 1)
        if D2:
            ks = torch.cat([ks, k2[k0[i] : k0[i] + n].double()[:, None].expand(n, H, D2)], -1)
        vs = v[k0[i] : k0[i] + n].double().view(n, G, -1)[..., :DV]
        vs = vs.expand(n, H, DV) if shared else vs.repeat_interleave(rep, 1)
        qs = q[rows].double().view(new[i], H, D1 + D2)
        s = (qs[:, None] * ks[None]).sum(-1).permute(0, 2, 1) * scale  # [new, H, n]
        mag = ((qs[:, None] * ks[None]).abs().sum(-1).permute(0, 2, 1) * scale).amax()
        at = past[i] + torch.arange(new[i], device="cuda")[:, None]
        j = torch.arange(n, device="cuda")[None]
        lo = torch.zeros_like(at)
        if window:
            lo = torch.maximum(lo, at - window + 1)
        if chunk:
            lo = torch.maximum(lo, at // chunk * chunk)
        see = (j <= at) & ((j >= lo) | (j < keep))
        if cap:
            s = cap * torch.tanh(s / cap)
        if slope is not None:
            s = s - slope.double()[None, :, None] * (at - j)[:, None]
        if sig is not None:
            p = torch.sigmoid(s + sig.double()[None, :, None]) * see[:, None]
        else:
            s = s.masked_fill(~see[:, None], float("-inf"))
            if sink is not None:
                s = torch.cat([s, sink.double()[None, :, None].expand(new[i], H, 1)], -1)
            p = torch.softmax(s, -1)[..., :n]
        want = (p.permute(0, 2, 1)[..., None] * vs[None]).sum(1)
        size = (p.permute(0, 2, 1)[..., None] * vs[None].abs()).sum(1)
        if gate is not None:
            f = torch.sigmoid(gate[rows].double().view(new[i], H, DV))
            want, size = want * f, size * f
        err = 2 * EPS * (n + mag * (D1 + D2 + 4) + 64) * size
        assert bool(((got[rows].double().view(new[i], H, DV) - want).abs() <= err + 1e-30).all())


def _fp32_path(S, q, k1, k2, v, out, H, hm, D1, D2, DV, shared, desc, max_new, scale, rep, window, keep, cap, sink, chunk, sig, slope, gate):
    """The fp32 products for either type of the keys (the launcher takes the matrix pipe for bf16 ones)."""
    L = S.L
    L.call("mi355_latent_attn", desc[0].numel(), max_new, H, hm, D1, D2, DV, L.ptr(q), q.stride(0), D1 + D2, L.ptr(k1), k1.stride(0), 0 if shared else D1, L.ptr(k2), 0 if k2 is None else k2.stride(0),
           L.ptr(v), v.stride(0), 0 if shared else (D1 if v is k1 else DV), L.ptr(out), out.stride(0), DV, S._dt(v), *[L.ptr(t) for t in desc], float(scale), 0, 1, None, 0, rep, window, keep, cap, L.ptr(sink),
           0, None, None, 0, None, chunk, L.ptr(sig), S._dt(out), L.ptr(slope), L.ptr(gate), 0 if gate is None else gate.stride(0))
    return out


@pytest.mark.parametrize("H,dk,dv,fixed,dt", [(1, 1, 5, False, F32), (2, 16, 64, False, BF16), (2, 17, 65, True, F32), (1, 64, 64, False, F32), (2, 96, 100, False, BF16), (1, 112, 64, True, F32), (1, 128, 130, False, F32), (1, 144, 64, True, BF16),
                                              (1, 256, 70, False, F32)])
def test_gla_in_groups_of_16_and_of_8_tokens(H, dk, dv, fixed, dt):
    """Key channels that fill the rows of 16 lanes and that do not, groups of 16 tokens and (where those exceed LDS or half the threads) of 8, sequences that end around a group.  The state
    rounds twice a token, the output dk + RC times: 64 bits within 2^-24 (2 T + dk + 40) of the sums of sizes (decays: a few roundings each, which the 16 T term holds)."""
    from llm_quest_amd import kernels_seq as S

    n = [1, 7, 8, 9, 0, 15, 16, 17, 33]
    T = sum(n)
    g = torch.Generator().manual_seed(dk + dv)
    q, k, v = (torch.randn(T, H * w, generator=g).to(dt).cuda() for w in (dk, dk, dv))
    z, bias, dec = torch.randn(T, H * dk, generator=g).cuda() + 2, 0.3 * torch.randn(H * dk, generator=g).cuda(), (0.5 + 0.5 * torch.rand(H, generator=g)).cuda()
    st0 = torch.randn(len(n) + 1, H, dk, dv, generator=g).cuda()
    slots = torch.arange(len(n), 0, -1)
    st = st0.clone()
    offs = [sum(n[:i]) for i in range(len(n) + 1)]
    if fixed:
        got = S.gla(q, k, v, None, None, 1.0, dk**-0.5, i32(offs), i32(slots.tolist()), st, H, dk, dv, head_decay=dec, kscale=0.5)
    else:
        got = S.gla(q, k, v, z, bias, 0.25, dk**-0.5, i32(offs), i32(slots.tolist()), st, H, dk, dv)
    a = dec.double()[None, :, None].expand(T, H, dk) if fixed else torch.sigmoid((z.double() + bias.double()).view(T, H, dk)) ** 0.25
    assert torch.equal(st[0], st0[0])
    for i, sl in enumerate(slots.tolist()):
        s, m = st0[sl].double(), st0[sl].double().abs()
        for t in range(offs[i], offs[i + 1]):
            kv = (k[t].double().view(H, dk, 1) * (0.5 if fixed else 1.0)) * v[t].double().view(H, 1, dv)
            s, m = a[t][..., None] * s + kv, a[t][..., None] * m + kv.abs()
            qt = q[t].double().view(H, dk) * dk**-0.5
            want, size = torch.einsum("hk,hkv->hv", qt, s), torch.einsum("hk,hkv->hv", qt.abs(), m)
            assert bool(((got[t].double().view(H, dv) - want).abs() <= EPS * (16 * (t - offs[i] + 1) + dk + 40) * size).all())
        assert bool(((st[sl].double() - s).abs() <= EPS * (16 * n[i] + 4) * m).all())


@pytest.mark.parametrize("M,K,N", [(1, 8, 7), (1, 1024, 33), (2, 264, 130), (3, 1024, 1024), (5, 1000, 17), (8, 2048, 2056), (6, 3072, 1025), (8, 512, 16400)])
def test_few_bf16_rows_with_a_bias(M, K, N):
    """Whole numbers whose sums fp32 holds exactly: the results are the exact sums rounded once; rows beside the operands and beside the bias are not read into them."""
    from llm_quest_amd import kernels_seq as S

    g = torch.Generator().manual_seed(M + K + N)
    x = torch.full((M + 1, K + 8), float("nan"), dtype=BF16, device="cuda")
    x[:M, :K] = torch.randint(-8, 9, (M, K), generator=g).cuda()
    w = torch.randint(-8, 9, (N, K), generator=g).to(BF16).cuda()
    bias = torch.randint(-999, 1000, (N,), generator=g).float().cuda()
    want = (x[:M, :K].double() @ w.double().T + bias.double()).float()
    for dt in (BF16, F32):
        assert torch.equal(S.linear(x[:M, :K], w, bias=bias, out_dtype=dt), want.to(dt))


@pytest.mark.parametrize("D,DV,window,cap,new,past", [(64, 64, 0, 0.0, [5, 130], [0, 70]), (128, 128, 100, 0.0, [1, 200, 17], [63, 0, 300]), (128, 40, 64, 5.0, [70, 3], [1, 400]), (256, 256, 0, 0.0, [9, 65], [120, 0]),
                                                      (72, 24, 50, 0.0, [33], [200]), (136, 136, 0, 2.0, [33], [200]), (128, 128, 0, 0.0, [1, 1], [4000, 2100]), (64, 64, 0, 0.0, [1], [600])])
def test_keys_of_one_part_and_of_two_give_the_same_attention(D, DV, window, cap, new, past):
    """Keys of one part come by their own loads (rows past the end are NaN here: they lie behind the descriptor's end), those of two parts by the general ones; queries at any
    alignment.  The arithmetic is the same, so are the bits.  One new token over many keys: up to 15 splits, more than the join requests at once.  Against 64 bits: queries, weights and
    results rounded to bf16 or held in it, 2^-9 each (a weight's error is its score's)."""
    from llm_quest_amd import kernels_seq as S

    H, half = 4, (D // 16) * 8
    g = torch.Generator().manual_seed(D + DV + window)
    total = [n + p for n, p in zip(new, past)]
    rows = [t + 70 for t in total]
    k, v = torch.full((sum(rows), D), float("nan")), torch.full((sum(rows), DV), float("nan"))
    at = [sum(rows[:i]) for i in range(len(rows))]
    for a, t in zip(at, total):
        k[a : a + t], v[a : a + t] = torch.randn(t, D, generator=g), torch.randn(t, DV, generator=g)
    k, v, q = k.to(BF16).cuda(), v.to(BF16).cuda(), torch.randn(sum(new), H * D, generator=g).cuda()
    shifted = torch.zeros(sum(new), H * D + 3, device="cuda")
    shifted[:, 1 : H * D + 1] = q
    k0, q0 = i32(at), i32([sum(new[:i]) for i in range(len(new))])
    desc = (q0, i32(new), i32(past), k0, k0, k0)

    def run(q, k1, k2, D1, D2):
        out = torch.full((sum(new), H * DV), float("nan"), device="cuda")
        S.latent_attn(q, k1, k2, v, out, H, H, D1, D2, DV, D, D1, DV, DV, desc, max(new), D**-0.5, max_keys=max(total), kv_rep=H, window=window, softcap=cap)
        return out

    one = run(q, k, None, D, 0)
    assert torch.equal(one, run(shifted[:, 1 : H * D + 1], k, None, D, 0))
    assert torch.equal(one, run(q, k[:, :half].contiguous(), k[:, half:].contiguous(), half, D - half))
    for i, (n, p) in enumerate(zip(new, past)):
        r = slice(int(q0[i]), int(q0[i]) + n)
        ks, vs, qs = k[at[i] : at[i] + n + p].double(), v[at[i] : at[i] + n + p].double(), q[r].double().view(n, H, D)
        s, mag = (qs @ ks.T) * D**-0.5, (qs.abs() @ ks.abs().T * D**-0.5).amax()
        s = cap * torch.tanh(s / cap) if cap else s
        pos, j = p + torch.arange(n, device="cuda")[:, None], torch.arange(n + p, device="cuda")[None]
        w = torch.softmax(s.masked_fill(((j > pos) | (j <= pos - (window or n + p + 1)))[:, None], float("-inf")), -1)
        err = (2.0**-8 * mag + 2.0**-8) * (w @ vs.abs()) + 1e-30
        assert bool(((one[r].double().view(n, H, DV) - w @ vs).abs() <= err).all())


@pytest.mark.parametrize("past", [700, 4000])
def test_what_is_not_finite_in_a_split_without_weight(past):
    """Keys whose weight is too small for a number still multiply their values: what is not finite there shows, whether a tile's keys are one split (no ``max_keys``) or several that are joined."""
    from llm_quest_amd import kernels_seq as S

    H, D, n = 4, 64, past + 1
    k, v, q = torch.full((n, D), -4.0), torch.randn(n, D, generator=torch.Generator().manual_seed(past)), torch.full((1, H * D), 4.0, device="cuda")
    k[:64] = 4.0  # all of the weight: the other scores are 369 powers of two below
    v[past - 40, 5], v[past - 40, 7], v[past - 41, 9] = float("nan"), float("inf"), float("-inf")
    k, v, zero = k.to(BF16).cuda(), v.to(BF16).cuda(), i32([0])
    out = []
    for keys in (0, n):
        o = torch.empty(1, H * D, device="cuda")
        S.latent_attn(q, k, None, v, o, H, H, D, 0, D, D, D, D, D, (zero, i32([1]), i32([past]), zero, zero, zero), 1, D**-0.5, max_keys=keys, kv_rep=H)
        out.append(o.view(H, D))
    assert S.attn_key_splits(1, 1, 1, H, n) > 1
    for o in out:
        assert bool(o[:, [5, 7, 9]].isnan().all()) and int(o.isnan().sum()) == 3 * H
    fine = [i for i in range(D) if i not in (5, 7, 9)]
    assert torch.allclose(out[0][:, fine], out[1][:, fine], rtol=2**-7, atol=1e-6)
