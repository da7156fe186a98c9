"""fp32 rows times bf16 weights on 64- and 128-row tiles (three bf16 products for one): ends of K, of rows and of columns, groups without rows, values that are not finite."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF16, F32 = torch.bfloat16, torch.float32


@pytest.mark.parametrize("K", [8, 16, 24, 32, 40, 64, 96, 128, 136, 264, 1000, 2048])
@pytest.mark.parametrize("M,N", [(65, 8), (129, 130), (450, 1024), (2100, 4100)])
def test_tiles_against_64_bits_and_the_kernel_of_few_rows(M, N, K):
    from llm_quest_amd import kernels_seq as S

    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x, w = torch.randn(M, K, generator=g, device="cuda"), torch.randn(N, K, generator=g, device="cuda").to(BF16)
    got = S.linear(x, w, out_dtype=F32)
    # eight runs of exact products, each run's and their sum's roundings: K + 8 of them at the most, of sums no larger than the magnitudes' sum
    bound = (K + 8) * 2.0**-24 * (x.double().abs() @ w.double().abs().T)
    assert bool(((got.double() - x.double() @ w.double().T).abs() <= bound).all())
    few = torch.tensor([0, M // 2, M - 1], device="cuda")
    assert torch.equal(S.linear(x[few].contiguous(), w, out_dtype=F32), got[few])  # a row's bits do not depend on the rows beside it


@pytest.mark.parametrize("sizes", [(70, 0, 1, 129), (64, 65, 0, 0), (1, 1, 200, 300)])
def test_tiles_of_groups_with_gathered_rows(sizes):
    from llm_quest_amd import kernels_seq as S

    T, N, K, E, top = sum(sizes), 200, 328, len(sizes), 2
    g = torch.Generator(device="cuda").manual_seed(T)
    x, w = torch.randn((T + 1) // 2, K, generator=g, device="cuda"), torch.randn(E, N, K, generator=g, device="cuda").to(BF16)
    x[0, 5] = float("inf")
    perm = torch.randperm(T, generator=g, device="cuda").to(torch.int32)
    offs = torch.tensor([0, *torch.tensor(sizes).cumsum(0).tolist()], dtype=torch.int32, device="cuda")
    out = torch.full((T, N), 7.0, device="cuda")
    S.bgemm(x, w, out, T, N, K, batch=E, sbn=K, b_bs=N * K, grp_offs=offs, a_rows=perm, a_div=top)
    for e in range(E):
        lo, hi = int(offs[e]), int(offs[e + 1])
        rows = x[(perm[lo:hi] // top).long()]
        want, bound = rows.double() @ w[e].double().T, (K + 8) * 2.0**-24 * (rows.double().abs() @ w[e].double().abs().T)
        ok = torch.isfinite(want)
        assert bool(((out[lo:hi].double() - want).abs() <= bound)[ok].all()) and torch.equal(out[lo:hi].double()[~ok], want[~ok])
