"""NT products of too few 256x256 tiles (one workgroup per CU, a ring of four K-tiles, row panels of 128 or 192): against 64 bits, and the bits of the 128x128 kernel (tile hint 1)."""

import pytest
import torch

from llm_quest_amd import _lib as L

pytestmark = pytest.mark.gpu
BF16, F32 = torch.bfloat16, torch.float32


def product(A, B, odt, bias=None, residual=None, hint=0, ldc=None, ws=True):
    M, N = A.shape[0], B.shape[0]
    C = torch.full((M, ldc or N), 7.0, dtype=odt, device="cuda")
    R = residual
    buf = torch.empty(32 << 20, dtype=F32, device="cuda") if ws else None
    L.require_gpu(A, B, C, bias, R, buf)
    L.call("mi355_gemm_bf16", L.GEMM_NT, M, N, A.shape[1], A.data_ptr(), A.stride(0), B.data_ptr(), B.stride(0), C.data_ptr(), C.stride(0), L.dt_code(odt), L.ptr(bias), L.ptr(R),
           R.stride(0) if R is not None else 0, 0, L.ptr(buf), buf.numel() * 4 if ws else 0, hint)
    if ldc:
        assert torch.equal(C[:, N:], torch.full_like(C[:, N:], 7.0))  # nothing beyond the matrix
    return C[:, :N]


def error_bound(A, B, extra):
    """Largest error of one fp32 sum of K exact bf16 products: K rounding steps of the sum of magnitudes (any order), and of what is added to it."""
    mag = A.double().abs() @ B.double().abs().t() + extra
    return (A.shape[1] + 4) * 2.0 ** -24 * mag


# one tile and parts of it; row panels of 128 and of 192 (5 100 x 1 024: 216 tiles of 192 rows, 320 of 128); the ring filled once, odd and even counts of K-tiles, a remainder in the last; K shares
# (long K, few tiles); 256 tiles of 192 rows where there are 128 of 256 x 256; without the ring (rows 0): more tiles than the one round, fewer K-tiles than the ring
SIZES = [(1, 8, 256, 128), (9, 16, 200, 128), (127, 128, 320, 128), (129, 136, 192, 0), (191, 264, 264, 128), (300, 1000, 1016, 128), (61, 1024, 3072, 128), (333, 1024, 3584, 128), (5100, 1024, 328, 192),
         (300, 16384, 256, 192), (2000, 4096, 256, 0), (300, 16392, 256, 0), (996, 768, 1992, 128)]


@pytest.mark.parametrize("M,N,K,rows", SIZES)
@pytest.mark.parametrize("odt", [BF16, F32])
@pytest.mark.parametrize("bias,residual", [(False, False), (True, True), (False, True)])
def test_against_64_bits(M, N, K, rows, odt, bias, residual):
    may_split = not bias and N % 8 == 0
    assert (L.load().mi355_gemm_nt_ring(M, N, K, L.dt_code(odt), may_split, 128 << 20) & 255) == rows
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    A = torch.randn(M, K, generator=g, device="cuda").to(BF16)
    B = torch.randn(N, K, generator=g, device="cuda").to(BF16)
    b = torch.randn(N, generator=g, device="cuda") if bias else None
    r = torch.randn(M, N, generator=g, device="cuda").to(odt) if residual else None
    got = product(A, B, odt, b, r)
    extra = (b.double() if bias else 0) + (r.double() if residual else 0)
    exact = A.double() @ B.double().t() + extra
    bound = error_bound(A, B, extra.abs() if bias or residual else 0)
    if odt == BF16:
        bound = bound + 2.0 ** -8 * exact.abs()  # one rounding to eight bits
    assert ((got.double() - exact).abs() <= bound).all()
    if K < 2048:  # no K shares, or the same: every sum in the same order
        assert torch.equal(product(A, B, odt, b, r, hint=1), got)


@pytest.mark.parametrize("odt", [BF16, F32])
@pytest.mark.parametrize("N,ldc,lda,skip", [(130, 133, 0, 0), (136, 140, 8, 0), (100, 100, 24, 3), (1024, 1025, 8, 1)])
def test_rows_that_are_not_aligned(N, ldc, lda, skip, odt):
    """Output and residual rows at any element, operands with longer rows, columns that end inside eight; nothing is written outside."""
    M, K = 150, 648
    g = torch.Generator(device="cuda").manual_seed(N)
    A = torch.randn(M, K + lda, generator=g, device="cuda").to(BF16)[:, :K]
    B = torch.randn(N, K + lda, generator=g, device="cuda").to(BF16)[:, :K]
    r = torch.randn(M, N + skip, generator=g, device="cuda").to(odt)[:, skip:]
    got, exact = product(A, B, odt, residual=r, ldc=ldc), A.double() @ B.double().t() + r.double()
    bound = error_bound(A, B, r.double().abs()) + (2.0 ** -8 * exact.abs() if odt == BF16 else 0)
    assert ((got.double() - exact).abs() <= bound).all()


@pytest.mark.parametrize("ws", [True, False])
def test_values_that_are_not_finite_stay_in_their_row(ws):
    assert (L.load().mi355_gemm_nt_ring(200, 256, 2048, L.dt_code(F32), ws, 128 << 20) >> 8 > 1) is ws
    A, B = torch.ones(200, 2048, device="cuda", dtype=BF16), torch.ones(256, 2048, device="cuda", dtype=BF16)
    A[3, 5], A[150, 2047], B[100, 64] = float("nan"), float("inf"), float("inf")
    got, want = product(A, B, F32, ws=ws), A.double() @ B.double().t()
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))
    assert torch.equal(got[torch.isfinite(got)], want[torch.isfinite(want)].float())


def test_same_bits_every_time():
    A, B = torch.randn(700, 3072, device="cuda").to(BF16), torch.randn(1024, 3072, device="cuda").to(BF16)
    first = product(A, B, BF16)
    assert all(torch.equal(first, product(A, B, BF16)) for _ in range(3))


@pytest.mark.parametrize("M,N,K", [(1279, 1024, 2048), (1280, 1024, 2048), (1280, 1024, 2040), (1500, 328, 3000), (4095, 1024, 4096), (1300, 64, 16392), (1300, 2048, 4096), (2000, 3072, 6144), (1300, 1024, 16328), (1300, 1024, 16320)])
def test_input_gradients_on_both_sides_of_the_rule(M, N, K):
    """dX = dY W by the NN form or on the transposed weight: the same product."""
    from llm_quest_amd import kernels as KK

    g = torch.Generator(device="cuda").manual_seed(M + K)
    dy, w = torch.randn(M, K, generator=g, device="cuda").to(BF16), torch.randn(K, N, generator=g, device="cuda").to(BF16)
    exact = dy.double() @ w.double()
    bound = error_bound(dy, w.t(), 0) + 2.0 ** -8 * exact.abs()
    assert ((KK.dgrad(dy, w).double() - exact).abs() <= bound).all()
    out = torch.empty(M, N, dtype=BF16, device="cuda")
    assert torch.equal(KK.dgrad(dy, w, out=out), KK.dgrad(dy, w))


@pytest.mark.parametrize("M,N,K,odt", [(300, 200, 320, BF16), (5100, 1000, 328, BF16), (5100, 1000, 328, F32), (129, 136, 256, F32)])
def test_a_residual_that_the_result_overwrites(M, N, K, odt):
    """Residual rows are read ahead of the rows that are written: the same result in place."""
    assert L.load().mi355_gemm_nt_ring(M, N, K, L.dt_code(odt), 1, 0)
    g = torch.Generator(device="cuda").manual_seed(M)
    A, B = (torch.randn(n, K, generator=g, device="cuda").to(BF16) for n in (M, N))
    r = torch.randn(M, N, generator=g, device="cuda").to(odt)
    apart = product(A, B, odt, residual=r)
    L.require_gpu(A, B, r)
    L.call("mi355_gemm_bf16", L.GEMM_NT, M, N, K, A.data_ptr(), K, B.data_ptr(), K, r.data_ptr(), N, L.dt_code(odt), None, r.data_ptr(), N, 0, None, 0, 0)
    assert torch.equal(r, apart)


@pytest.mark.parametrize("M,N,K,shares", [(2000, 1024, 4096, 1), (996, 1024, 4096, 2), (333, 1024, 3584, 8), (700, 512, 8192, 8), (1300, 1536, 6144, 1), (5664, 1024, 3584, 1), (12, 32000, 2048, 1), (1000, 3000, 2056, 1)])
@pytest.mark.parametrize("residual", [False, True])
def test_fp32_results_are_no_further_from_64_bits(M, N, K, shares, residual):
    """A sum in fewer shares is longer and rounds more; fp32 results would show it: where the ring takes fewer it cuts them in its workgroups.  The 128 x 128 kernel with its own shares (hint 1) is the
    measure: one per cent for the spread of a norm over a third of a million results and more (a residual of their size, once added, rounds both alike)."""
    rows = L.load().mi355_gemm_nt_ring(M, N, K, L.dt_code(F32), 1, 128 << 20)
    assert rows >> 8 >= shares
    g = torch.Generator(device="cuda").manual_seed(M + K)
    A, B = (torch.randn(n, K, generator=g, device="cuda").to(BF16) for n in (M, N))
    r = torch.randn(M, N, generator=g, device="cuda") if residual else None
    exact = A.double() @ B.double().t() + (r.double() if residual else 0)
    err = [float((product(A, B, F32, residual=r, hint=h).double() - exact).norm()) for h in (0, 1)]
    assert err[0] <= 1.01 * err[1]


# ---- the NN form: one tile and parts of it, panels of 128 and of 192 rows, the ring filled once, odd and even counts of K-tiles, a remainder in the last, K shares
NN_SIZES = [(1, 8, 256, 128), (9, 16, 200, 128), (127, 128, 320, 128), (129, 136, 192, 0), (191, 264, 264, 128), (300, 1000, 1016, 128), (61, 1024, 3072, 128), (333, 1024, 3584, 128), (5100, 1024, 328, 192),
            (300, 16384, 256, 192), (2000, 4096, 256, 0), (996, 768, 1992, 128), (4096, 1024, 448, 128), (61, 256, 66000, 128), (197, 256, 66000, 0), (602, 128, 33000, 0)]


@pytest.mark.parametrize("M,N,K,rows", NN_SIZES)
@pytest.mark.parametrize("odt", [BF16, F32])
@pytest.mark.parametrize("bias,residual", [(False, False), (True, True)])
def test_nn_against_64_bits(M, N, K, rows, odt, bias, residual):
    if not bias:
        assert (L.load().mi355_gemm_nn_ring(M, N, K, L.dt_code(odt), 1, 128 << 20) & 255) == rows
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    A = torch.randn(M, K + 8, generator=g, device="cuda").to(BF16)[:, :K]
    W = torch.randn(K, N + 16, generator=g, device="cuda").to(BF16)[:, 8 : N + 8]  # rows longer than the operand: nothing beside it is read into a sum
    b = torch.randn(N, generator=g, device="cuda") if bias else None
    r = torch.randn(M, N, generator=g, device="cuda").to(odt) if residual else None

    def take(hint):
        C, buf = torch.full((M, N + 4), 7.0, dtype=odt, device="cuda"), torch.empty(32 << 20, dtype=F32, device="cuda")
        L.require_gpu(A, W, C, b, r, buf)
        L.call("mi355_gemm_bf16", L.GEMM_NN, M, N, K, A.data_ptr(), A.stride(0), W.data_ptr(), W.stride(0), C.data_ptr(), C.stride(0), L.dt_code(odt), L.ptr(b), L.ptr(r), N if residual else 0, 0, buf.data_ptr(),
               buf.numel() * 4, hint)
        assert torch.equal(C[:, N:], torch.full_like(C[:, N:], 7.0))
        return C[:, :N]

    got, extra = take(0), (b.double() if bias else 0) + (r.double() if residual else 0)
    exact = A.double() @ W.double() + extra
    bound = error_bound(A, W.t(), extra.abs() if bias or residual else 0)
    if odt == BF16:
        bound = bound + 2.0 ** -8 * exact.abs()  # one rounding to eight bits
    assert ((got.double() - exact).abs() <= bound).all()
    if K < 2048:  # no K shares, or the same: every sum in the same order
        assert torch.equal(take(1), got)


@pytest.mark.parametrize("M,N,K", [(333, 1024, 3584), (996, 1024, 6144), (2000, 1024, 4096), (197, 768, 2304)])
def test_nn_fp32_results_are_no_further_from_64_bits(M, N, K):
    """As for the NT form: the 128 x 128 kernel with its own shares of K (hint 1) is the measure."""
    assert L.load().mi355_gemm_nn_ring(M, N, K, L.dt_code(F32), 1, 128 << 20)
    g = torch.Generator(device="cuda").manual_seed(M + K)
    A, W = torch.randn(M, K, generator=g, device="cuda").to(BF16), torch.randn(K, N, generator=g, device="cuda").to(BF16)
    exact, buf, err = A.double() @ W.double(), torch.empty(32 << 20, dtype=F32, device="cuda"), []
    for hint in (0, 1):
        C = torch.empty(M, N, device="cuda")
        L.require_gpu(A, W, C, buf)
        L.call("mi355_gemm_bf16", L.GEMM_NN, M, N, K, A.data_ptr(), K, W.data_ptr(), N, C.data_ptr(), N, L.dt_code(F32), None, None, 0, 0, buf.data_ptr(), buf.numel() * 4, hint)
        err.append(float((C.double() - exact).norm()))
    assert err[0] <= 1.01 * err[1]


def test_nn_values_that_are_not_finite_stay_in_their_row_and_column():
    A, W = torch.ones(200, 2048, device="cuda", dtype=BF16), torch.ones(2048, 256, device="cuda", dtype=BF16)
    A[3, 5], A[150, 2047], W[64, 100] = float("nan"), float("inf"), float("inf")
    from llm_quest_amd import kernels as KK

    got, want = KK.gemm(L.GEMM_NN, A, W, out_dtype=F32), A.double() @ W.double()
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))
    assert torch.equal(got[torch.isfinite(got)], want[torch.isfinite(want)].float())


@pytest.mark.parametrize("M,N,K,rows", [(1, 8, 256, 128), (127, 128, 320, 128), (333, 3072, 1024, 128), (5100, 1000, 328, 192), (129, 136, 192, 0), (2000, 3072, 256, 0)])
def test_fused_epilogues_are_the_128_x_128_kernels(M, N, K, rows):
    """SwiGLU's backward behind the NN form, GELU (with and without a residual) behind the NT form: the bits of hint 1, rows and columns that end inside a tile, nothing written beside them."""
    lib, g = L.load(), torch.Generator(device="cuda").manual_seed(M + N)
    assert lib.mi355_gemm_nn_ring(M, N, K, 0, 0, 0) & 255 == rows
    A, W = torch.randn(M, K, generator=g, device="cuda").to(BF16), (torch.randn(K, N, generator=g, device="cuda") * 0.1).to(BF16)
    gu, Wt = torch.randn(M, 2 * N + 16, generator=g, device="cuda").to(BF16)[:, 8 : 2 * N + 8], W.t().contiguous()
    r, bias = torch.randn(M, N, generator=g, device="cuda").to(BF16), torch.randn(N, generator=g, device="cuda")

    def take(form, b, width, residual, epi, hint, bias=None):
        C = torch.full((M, width + 8), 7.0, dtype=BF16, device="cuda")
        L.require_gpu(A, b, C, residual, bias)
        L.call("mi355_gemm_bf16", form, M, N, K, A.data_ptr(), K, b.data_ptr(), b.stride(0), C.data_ptr(), C.stride(0), L.DT_BF16, L.ptr(bias), L.ptr(residual), 0 if residual is None else residual.stride(0), epi, None, 0, hint)
        assert torch.equal(C[:, width:], torch.full_like(C[:, width:], 7.0))
        return C[:, :width]

    assert torch.equal(take(L.GEMM_NN, W, 2 * N, gu, L.EPI_SWIGLU_BWD, 0), take(L.GEMM_NN, W, 2 * N, gu, L.EPI_SWIGLU_BWD, 1))
    for residual in (None, r):
        assert torch.equal(take(L.GEMM_NT, Wt, N, residual, L.EPI_GELU, 0, bias), take(L.GEMM_NT, Wt, N, residual, L.EPI_GELU, 1, bias))


@pytest.mark.parametrize("M,F_,K", [(1, 32, 256), (127, 64, 320), (130, 96, 1000), (333, 3584, 1024), (257, 416, 328), (5100, 480, 328), (1056, 3584, 512)])
def test_swiglu_forward_is_the_128_x_128_kernels(M, F_, K):
    """Gate-up rows and activations have the bits of hint 1 and of the product and ``swiglu_fwd`` by themselves; rows, units (32 of a tile's 64) and K end inside a tile; nothing beside either is written."""
    from llm_quest_amd import kernels as KK

    g = torch.Generator(device="cuda").manual_seed(M + F_)
    A, W = torch.randn(M, K, generator=g, device="cuda").to(BF16), (torch.randn(2 * F_, K + 8, generator=g, device="cuda") * 0.1).to(BF16)[:, :K]

    def take(hint):
        C, act = torch.full((M + 1, 2 * F_ + 8), 7.0, dtype=BF16, device="cuda"), torch.full((M + 1, F_ + 8), 7.0, dtype=BF16, device="cuda")
        L.call("mi355_gemm_bf16", L.GEMM_NT, M, 2 * F_, K, A.data_ptr(), K, W.data_ptr(), W.stride(0), C.data_ptr(), C.stride(0), L.DT_BF16, None, act.data_ptr(), act.stride(0), L.EPI_SWIGLU_FWD, None, 0, hint)
        assert all(bool((x[M:] == 7).all()) and bool((x[:, n:] == 7).all()) for x, n in ((C, 2 * F_), (act, F_)))
        return C[:M, : 2 * F_], act[:M, :F_]

    (gu, act), (want_gu, want_act) = take(0), take(1)
    assert torch.equal(gu, want_gu) and torch.equal(act, want_act)
    assert torch.equal(act, KK.swiglu_fwd(gu.contiguous(), F_))


@pytest.mark.parametrize("tokens", [32, 33, 64, 96, 97, 500, 1000])
def test_wide_weight_gradients_of_few_tokens(tokens):
    """Gradients of a thousand 256 x 256 tiles: the two tiles that a short sum may take give the same bits, which are the fp32 sum rounded once."""
    from llm_quest_amd import _lib as L

    V, D = 65536 + 40, 1024
    g = torch.Generator().manual_seed(tokens)
    dy, x = torch.randn(tokens, V, generator=g).to(torch.bfloat16).cuda(), torch.randn(tokens, D, generator=g).to(torch.bfloat16).cuda()
    outs = []
    for hint in (0, 2, 3):
        out = torch.empty(V, D, dtype=torch.bfloat16, device="cuda")
        L.require_gpu(dy, x, out)
        L.call("mi355_gemm_bf16", 2, V, D, tokens, L.ptr(dy), V, L.ptr(x), D, L.ptr(out), D, L.DT_BF16, None, None, 0, 0, None, 0, hint)
        outs.append(out)
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    want = dy[:, -300:].float().T.contiguous() @ x.float()
    assert float((outs[0][-300:].float() - want).norm()) < 2**-8 * float(want.norm())
