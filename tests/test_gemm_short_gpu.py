"""NT products of short sums over many tiles (csrc/gemm_persist.h): the bits of the eight-wave tile (hint 2), which has its own tests against 64 bits, and which sums take it."""

import pytest
import torch

from llm_quest_amd import _lib as L
from llm_quest_amd import kernels as K

pytestmark = pytest.mark.gpu
BF16, F32 = torch.bfloat16, torch.float32


def draw(seed, *shape, dtype=BF16):
    return torch.randn(*shape, generator=torch.Generator(device="cuda").manual_seed(seed), device="cuda").to(dtype)


def kernels_of(fn):
    fn()
    torch.cuda.synchronize()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as p:
        fn()
        torch.cuda.synchronize()
    return {e.key for e in p.key_averages()}


# two K-tiles and more, odd and even numbers of them; rows and columns that end inside a tile, more tiles than CUs (a workgroup walks two or three), more than 128 column panels (their own walk; panels that are no multiple of four)
@pytest.mark.parametrize("M,N,K_", [(300, 264, 128), (513, 776, 192), (2049, 1288, 256), (33_001, 776, 320), (12_000, 2056, 192), (16_640, 2048, 512), (300, 33_288, 128), (700, 33_800, 320)])
def test_bits_of_the_eight_wave_tile(M, N, K_, monkeypatch):
    monkeypatch.setenv("MI355_GEMM_PERSIST_MIN_TILES", "1")
    x, w, res = draw(M, M, K_ + 8)[:, :K_], draw(N, N, K_), draw(3, M, N)
    wide = torch.full((M + 1, N + 8), 7.0, dtype=BF16, device="cuda")
    K.gemm(L.GEMM_NT, x, w, out=wide[:M, :N], allow_split_k=False)
    assert bool((wide[M:] == 7).all()) and bool((wide[:, N:] == 7).all())
    assert torch.equal(wide[:M, :N], K.gemm(L.GEMM_NT, x, w, tile=2, allow_split_k=False))
    assert torch.equal(K.gemm(L.GEMM_NT, x, w, residual=res, allow_split_k=False), K.gemm(L.GEMM_NT, x, w, residual=res, tile=2, allow_split_k=False))
    F = N // 64 * 32
    for a, b in zip(K.gemm_gateup_swiglu(x, w[: 2 * F]), K.gemm_gateup_swiglu(x, w[: 2 * F], tile=2)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("K_,plain,gateup,residual", [(128, True, True, True), (192, True, True, True), (256, True, True, False), (320, True, True, False), (512, True, False, False), (576, True, True, False),
                                                      (640, False, False, False), (704, True, True, False), (768, False, False, False), (832, True, False, False), (896, False, False, False), (960, False, False, False)])
def test_which_sums_take_it(K_, plain, gateup, residual):
    M, N = 16_384, 2048  # 512 tiles; under them, and where the caller keeps persistent kernels off, none does
    x, w, res = draw(1, M, K_), draw(2, N, K_), draw(3, M, N)
    took = lambda fn: any("gemm_nt_persist_kernel" in n for n in kernels_of(fn))
    assert took(lambda: K.gemm(L.GEMM_NT, x, w)) is plain
    assert took(lambda: K.gemm_gateup_swiglu(x, w)) is gateup
    assert took(lambda: K.gemm(L.GEMM_NT, x, w, residual=res)) is residual
    assert not took(lambda: K.gemm(L.GEMM_NT, x[: M - 256], w))
    if K_ in (128, 320, 640):
        wn = draw(2, K_, N)
        assert took(lambda: K.dgrad(x, wn)) is plain and K.dgrad_on_quad(M, N, K_) is not plain
        K.persistent_gemm(False)
        try:
            assert not took(lambda: K.gemm(L.GEMM_NT, x, w))
        finally:
            K.persistent_gemm(True)


@pytest.mark.parametrize("B,S,Hq", [(6, 709, 4), (9, 500, 3)])
@pytest.mark.parametrize("K_", [128, 192, 256, 320, 384, 448])
def test_attention_constants_behind_short_sums(B, S, Hq, K_, monkeypatch):
    """d(ctx) in the bits of the plain product, its row sums with ctx per head (128 products of 16-bit numbers in fp32, in any order), their negatives and the scaled lse in the backward's scratch; an odd
    number of heads, rows that end inside a tile.  384 is four waves' (csrc/gemm.hip: short_nt)."""
    monkeypatch.setenv("MI355_GEMM_PERSIST_MIN_TILES", "1")
    dy, w, ctx, lse = draw(1, B * S, K_), draw(2, K_, Hq * 128), draw(3, B * S, Hq * 128), draw(4, B, Hq, S, dtype=F32)
    fn = lambda: K.dgrad_attn_delta(dy, w, ctx, lse, B, S, Hq, 128)
    dctx, delta = fn()
    assert any("gemm_nt_persist_kernel" in n for n in kernels_of(fn)) is (K_ != 384)
    assert torch.equal(dctx, K.gemm(L.GEMM_NT, dy, w.T.contiguous(), tile=2, allow_split_k=False))
    prod = (dctx.double() * ctx.double()).view(B, S, Hq, 128).permute(0, 2, 1, 3)
    assert bool(((delta.double() - prod.sum(-1)).abs() <= 128 * 2.0**-24 * prod.abs().sum(-1)).all())
    lib, n = L.load(), 4 * B * Hq * S
    ws = K._attn_scratch(dy.device, lib.mi355_attn_bwd_workspace_bytes(B, S, Hq, 128))
    nl2, ndl = (ws[o : o + n].view(F32).view(B, Hq, S) for o in (lib.mi355_attn_bwd_workspace_rowconst_offset(B, S, Hq, 128, i) for i in (0, 1)))
    assert torch.equal(ndl, -delta) and torch.equal(nl2, -lse * torch.tensor(1.4426950408889634, dtype=F32, device="cuda"))


def test_weight_gradients_just_beyond_one_round_of_tiles():
    """Few tokens: 128 x 128 tiles (in brackets those of 256 x 256) where they are one round of two a CU, and where the larger ones need a second round for a few."""
    def small(T, shapes, odt=BF16):
        pr = [(draw(1, T, m), draw(2, T, n), torch.empty(m, n, dtype=odt, device="cuda"), None) for m, n in shapes]
        fn = (lambda: K.gemm(L.GEMM_TN, pr[0][0], pr[0][1], out_dtype=odt)) if len(shapes) == 1 else (lambda: K.gemm_grouped(L.GEMM_TN, pr))
        return not any("gemm_quad" in n for n in kernels_of(fn))

    assert small(300, [(2304, 768), (768, 2048), (4112, 768), (768, 2056)])  # 504 (129)
    assert not small(300, [(2304, 768), (768, 2304), (4112, 768), (768, 2056)])  # 516 (132)
    assert small(640, [(8224, 2048)]) and small(640, [(8704, 2048)]) and not small(1024, [(8704, 2048)]) and small(300, [(9216, 2048)]) and not small(640, [(9216, 2048)]) and not small(300, [(9472, 2048)])  # (264, 272, 288, 296)
