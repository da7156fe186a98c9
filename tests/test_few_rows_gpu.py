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
