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
