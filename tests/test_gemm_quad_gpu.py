"""Products on 256x256 tiles by four waves of 128x128 (csrc/gemm_quad.h): the bits of the tiles that they took over from (tile hints 2 and 5), which have their own tests against 64 bits."""

import pytest
import torch

from llm_quest_amd import _lib as L
from llm_quest_amd import kernels as K

pytestmark = pytest.mark.gpu
BF16, F32 = torch.bfloat16, torch.float32


def draw(seed, *shape, dtype=BF16):
    return torch.randn(*shape, generator=torch.Generator(device="cuda").manual_seed(seed), device="cuda").to(dtype)


def nt(A, B, odt, bias, residual, hint, pad):
    M, N = A.shape[0], B.shape[0]
    C = torch.full((M + 1, N + pad), 7.0, dtype=odt, device="cuda")
    L.call("mi355_gemm_bf16", L.GEMM_NT, M, N, A.shape[1], L.ptr(A), A.stride(0), L.ptr(B), B.stride(0), L.ptr(C), C.stride(0), L.dt_code(odt), L.ptr(bias), L.ptr(residual),
           0 if residual is None else residual.stride(0), 0, None, 0, hint)
    assert bool((C[M:] == 7).all()) and bool((C[:, N:] == 7).all())  # nothing beyond the matrix
    return C[:M, :N]


# the shortest sum (four K-tiles), odd and even counts of K-tiles; one row, parts of a tile's rows and columns, whole tiles, more tiles than CUs (a workgroup walks two or three) with both parities
@pytest.mark.parametrize("M,N,K_", [(1, 256, 256), (257, 264, 320), (383, 520, 448), (512, 512, 576), (700, 8, 1024), (130, 1288, 2048), (33_000, 520, 256), (17_000, 1800, 320)])
@pytest.mark.parametrize("odt", [BF16, F32])
@pytest.mark.parametrize("bias,residual", [(False, False), (True, False), (False, True), (True, True)])
def test_nt_gives_the_bits_of_the_eight_wave_tile(M, N, K_, odt, bias, residual):
    A, B = draw(M, M, K_ + 8)[:, :K_], draw(N, N, K_)
    b = draw(3, N, dtype=F32) if bias else None
    r = draw(4, M, N + 16, dtype=odt)[:, :N] if residual else None
    assert torch.equal(nt(A, B, odt, b, r, 7, 8), nt(A, B, odt, b, r, 2, 8))


# weights as they lie: rows of A end inside a tile, columns of B too (its rows are K's, whole K-tiles); odd and even counts of K-tiles; more tiles than CUs
@pytest.mark.parametrize("M,N,K_", [(1, 256, 256), (257, 264, 320), (383, 520, 448), (512, 512, 576), (700, 8, 1024), (130, 1288, 2048), (33_000, 520, 256), (17_000, 1800, 320)])
@pytest.mark.parametrize("kind", ["plain", "residual", "swiglu"])
def test_nn_gives_the_bits_of_the_eight_wave_tile(M, N, K_, kind):
    A, B, W = draw(M, M, K_ + 8)[:, :K_], draw(N, K_, N + 24)[:, :N], 2 * N if kind == "swiglu" else N
    r = None if kind == "plain" else draw(4, M, W + 16)[:, :W]

    def take(hint):
        C = torch.full((M + 1, W + 8), 7.0, dtype=BF16, device="cuda")
        L.call("mi355_gemm_bf16", L.GEMM_NN, M, N, K_, L.ptr(A), A.stride(0), L.ptr(B), B.stride(0), L.ptr(C), C.stride(0), L.DT_BF16, None, L.ptr(r), 0 if r is None else r.stride(0),
               L.EPI_SWIGLU_BWD if kind == "swiglu" else 0, None, 0, hint)
        assert bool((C[M:] == 7).all()) and bool((C[:, W:] == 7).all())
        return C[:M, :W]

    assert torch.equal(take(7), take(2))


# the library's own choice of input gradients: a main part and a remainder on small tiles, long sums in shares of K (one tile in 32, eight, 32 and 192 tiles), plain and behind SwiGLU; against the transposed weight's product
@pytest.mark.parametrize("M,N,K_", [(4352, 3080, 256), (17016, 1024, 320), (2836, 3072, 1024), (256, 256, 20032), (333, 1024, 50304), (1300, 1000, 33024), (12100, 1000, 16448), (498, 2048, 16384)])
def test_input_gradients_of_weights_as_they_lie(M, N, K_):
    dy, w = draw(M, M, K_), draw(N, K_, N) * K_**-0.5
    wt = w.T.contiguous()
    got, want = K.dgrad(dy, w), dy.double() @ w.double() if M * K_ < 1e8 else None
    assert off(got, K.gemm(L.GEMM_NT, dy, wt, out_dtype=F32), K_, BF16)
    if want is not None:
        assert off(got, want, K_, BF16)
    if K_ <= 1024:
        assert K.dgrad_on_quad(M, N, K_)
        # (17 016 rows are cut: whole rounds of 256 tiles, and a remainder on small tiles whose sums are cut in either form)
        main = M if M != 17016 else 256 // ((N + 255) // 256) * 256
        assert torch.equal(got[:main], K.gemm(L.GEMM_NT, dy[:main], wt, allow_split_k=False))
        if main < M:  # row by row: a few wrong ones at the seam are off by their size
            want = dy[main:].double() @ w.double()
            assert float(((got[main:].double() - want).norm(dim=1) / want.norm(dim=1)).max()) < 2**-24 * K_**0.5 + 2**-8
        gu = draw(7, M, 2 * N)
        assert torch.equal(K.gemm_dgrad_swiglu_bwd(dy, w, gu), K.swiglu_bwd(gu, K.gemm(L.GEMM_NN, dy, w, allow_split_k=False), N))


# K = tokens: the shortest, remainders of one row and of all but one in the last K-tile, odd and even counts; columns that end inside a tile; more tiles than CUs
@pytest.mark.parametrize("M,N,K_", [(256, 256, 193), (264, 520, 257), (512, 256, 1024), (1000, 1288, 639), (2048, 8, 705), (4104, 4360, 321)])
@pytest.mark.parametrize("odt", [BF16, F32])
@pytest.mark.parametrize("residual", [False, True])
def test_tn_gives_the_bits_of_the_four_wave_tile_of_short_k_tiles(M, N, K_, odt, residual):
    A, B = draw(M, K_, M + 8)[:, :M], draw(N, K_, N)
    r = draw(4, M, N, dtype=odt) if residual else None

    def take(hint):
        C = torch.full((M + 1, N + 8), 7.0, dtype=odt, device="cuda")
        L.call("mi355_gemm_bf16", L.GEMM_TN, M, N, K_, L.ptr(A), A.stride(0), L.ptr(B), N, L.ptr(C), N + 8, L.dt_code(odt), None, L.ptr(r), N if residual else 0, 0, None, 0, hint)
        assert bool((C[M:] == 7).all()) and bool((C[:, N:] == 7).all())
        return C[:M, :N]

    assert torch.equal(take(7), take(5))


# the library's own choice of a layer's weight gradients: 160 tiles and more in one launch, a residual on one problem only; tokens that end inside a K-tile
@pytest.mark.parametrize("tokens", [1025, 2048])
@pytest.mark.parametrize("odt", [BF16, F32])
def test_grouped_weight_gradients(tokens, odt):
    shapes = [(2048, 1024), (1024, 3080), (6144, 1024), (264, 776)]
    problems = []
    for i, (m, n) in enumerate(shapes):
        problems.append((draw(i, tokens, m), draw(9 + i, tokens, n), torch.empty(m, n, dtype=odt, device="cuda"), draw(20, m, n, dtype=odt) if i == 1 else None))
    K.gemm_grouped(L.GEMM_TN, problems)
    for a, b, out, r in problems:
        assert torch.equal(out, K.gemm(L.GEMM_TN, a, b, out_dtype=odt, residual=r, allow_split_k=False, tile=5))


def off(got, want, terms, odt):
    """Relative error of sums of `terms` products within what fp32 sums (and a bf16 result: eight significant bits) are off by."""
    got, want = got.double(), want.double()
    return float((got - want).norm() / want.norm()) < 2**-24 * terms**0.5 + (2**-8 if odt == BF16 else 0)


# few tiles of long sums: shares of K, added up by a second kernel.  K = 64 n of every remainder of shares; rows, columns and (TN) K that end inside a tile; one tile in sixteen shares, several rounds of the CUs
@pytest.mark.parametrize("form,M,N,K_", [("nt", 257, 264, 4096), ("nt", 5664, 1024, 12288), ("nt", 8100, 1024, 8256), ("nt", 300, 520, 16448), ("nt", 12100, 1000, 33024),
                                         ("tn", 264, 256, 4097), ("tn", 1000, 1288, 8191), ("tn", 3072, 768, 5664), ("tn", 6144, 1024, 5665), ("tn", 2304, 776, 12287)])
@pytest.mark.parametrize("odt", [BF16, F32])
@pytest.mark.parametrize("residual", [False, True])
def test_shares_of_k(form, M, N, K_, odt, residual):
    A, B = (draw(M, M, K_), draw(N, N, K_)) if form == "nt" else (draw(M, K_, M), draw(N, K_, N))
    C = torch.full((M + 1, N + 8), 7.0, dtype=odt, device="cuda")
    r = draw(4, M, N, dtype=odt) if residual else None
    K.gemm(L.GEMM_NT if form == "nt" else L.GEMM_TN, A, B, out=C[:M, :N], residual=r)
    assert bool((C[M:] == 7).all()) and bool((C[:, N:] == 7).all())
    rows = torch.cat([torch.arange(min(64, M)), torch.arange(max(0, M - 64), M)]).cuda()
    want = A[rows].double() @ B.double().T if form == "nt" else A[:, rows].double().T @ B.double()
    assert off(C[rows, :N], want + (r[rows].double() if residual else 0), K_, odt)


# a block's weight gradients in shares: alone, and behind a first launch that the others fill (332 tiles)
@pytest.mark.parametrize("tokens,shapes", [(4096, [(512, 512)] * 3), (5664, [(8256, 1024), (1024, 2048), (7168, 1024), (1024, 3584)]), (8191, [(2304, 768), (768, 776), (3072, 768)])])
@pytest.mark.parametrize("odt", [BF16, F32])
def test_shares_of_grouped_weight_gradients(tokens, shapes, odt):
    problems = []
    for i, (m, n) in enumerate(shapes):
        C = torch.full((m + 1, n + 8), 7.0, dtype=odt, device="cuda")
        problems.append((draw(i, tokens, m), draw(i + 9, tokens, n), C[:m, :n], draw(5, m, n, dtype=odt) if i == 1 else None, C))
    K.gemm_grouped(L.GEMM_TN, [q[:4] for q in problems])
    for a, b, c, r, whole in problems:
        assert bool((whole[c.shape[0] :] == 7).all()) and bool((whole[:, c.shape[1] :] == 7).all())
        want = a[:, -96:].double().T @ b.double()
        assert off(c[-96:], want + (r[-96:].double() if r is not None else 0), tokens, odt)


# rows of results in whole lines of 128 bytes (stored past the L2) and in parts of them: pitches that are a multiple of it and one that is not, a corner beside a line's start; columns that end inside a line
WHOLE = [("nt", 383, 520, 448), ("nt", 17_000, 1792, 320), ("tn", 520, 1288, 639), ("nn", 383, 520, 448), ("swiglu", 383, 544, 448), ("swiglu", 383, 520, 448), ("swiglu", 4000, 1088, 256), ("gateup", 600, 576, 320), ("gateup", 600, 512, 320)]


@pytest.mark.parametrize("form,M,N,K_,odt", [(*c, odt) for c in WHOLE for odt in (BF16, F32)[: 2 if c[0] in ("nt", "tn") else 1]])
def test_results_in_whole_lines_and_in_parts_of_them(form, M, N, K_, odt):
    A, B = (draw(M, K_, M), draw(N, K_, N)) if form == "tn" else (draw(M, M, K_), draw(N, K_, N) if form in ("nn", "swiglu") else draw(N, N, K_))
    gu, act = draw(4, M, 2 * N), torch.empty(M, N // 2, dtype=BF16, device="cuda")
    W = 2 * N if form == "swiglu" else N

    def take(hint, ld, first):
        C = torch.full((M + 1, ld), 7.0, dtype=odt, device="cuda")
        at = C[:M, first : first + W]
        L.call("mi355_gemm_bf16", {"nt": L.GEMM_NT, "gateup": L.GEMM_NT, "tn": L.GEMM_TN}.get(form, L.GEMM_NN), M, N, K_, L.ptr(A), A.stride(0), L.ptr(B), B.stride(0), L.ptr(at), ld, L.dt_code(odt), None,
               *{"swiglu": (L.ptr(gu), 2 * N, L.EPI_SWIGLU_BWD), "gateup": (L.ptr(act), N // 2, L.EPI_SWIGLU_FWD)}.get(form, (None, 0, 0)), None, 0, hint)
        assert bool((C[M:] == 7).all()) and bool((C[:, :first] == 7).all()) and bool((C[:, first + W :] == 7).all())
        return at

    want = take(5 if form == "tn" else 2, W, 0)
    whole = (W + 127) // 64 * 64  # of elements: whole lines in either type
    for ld, first in ((whole, 0), (whole + 64, 64), (whole, 8), (W + 8, 0), (W + 24, 16)):
        assert torch.equal(take(7, ld, first), want), (ld, first)
