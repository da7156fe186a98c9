"""Products of groups of rows on 256x256 tiles by four waves (csrc/bgemm_quad.h) against 64 bits."""

import pytest
import torch

from llm_quest_amd import kernels_seq as S

pytestmark = pytest.mark.gpu
BF16, F32 = torch.bfloat16, torch.float32

# rows of the groups: every number of 16-row blocks that a wave has a variant for and both sides of where the next one begins; groups of none, one and several tiles with a part of one left
EDGES = [1, 0, 15, 17, 31, 33, 63, 65, 0, 127, 129, 191, 193, 223, 225, 255, 256, 257, 300, 513, 0]
# the shortest sum (four K-tiles), longer ones; columns that end inside a tile and inside its first half; more tiles than CUs (a workgroup walks several of different heights)
CASES = [(EDGES, 1032, 256, 0, F32), (EDGES, 2568, 384, 0, BF16), (EDGES, 2560, 512, 1, F32), (EDGES, 1856, 256, 4, BF16), (EDGES, 2048, 640, 2, F32), (EDGES, 1216, 256, 3, BF16),
         ([1100, 0, 3, 700], 5000, 256, 0, BF16), ([2] * 250, 264, 256, 4, BF16), ([], 2056, 256, 1, BF16), ([], 4096, 384, 4, F32)]
# ... the same at the shortest sums that groups take the four waves for (bgemm.hip; under them the eight-wave kernel's): 768, SiLU 512, the other gated ones 1 280
CASES += [(EDGES, 1032, 768, 0, F32), (EDGES, 2568, 896, 0, BF16), (EDGES, 2560, 768, 1, F32), (EDGES, 1856, 512, 4, BF16), (EDGES, 2048, 1280, 2, F32), (EDGES, 1216, 1408, 3, BF16), ([1100, 0, 3, 700], 5000, 768, 0, BF16),
          ([2] * 250, 264, 512, 4, BF16)]


@pytest.mark.parametrize("lens,N,K,epi,odt", CASES)
def test_groups_of_rows(lens, N, K, epi, odt):
    g = torch.Generator(device="cuda").manual_seed(N + K)
    n = (N + 63) // 64 * 64 if epi >= 2 else N  # weight rows; of a gated product in blocks of 32 gate and 32 up rows
    width = (N // 2 - 8) // 8 * 8 if epi >= 2 else N
    batch, R, each = (len(lens), sum(lens), 0) if lens else (5, 5 * 700, 700)  # (no groups: five matrices of 700 rows)
    a = torch.randn(R, K + 8, generator=g, device="cuda").to(BF16)[:, :K]
    w = (torch.randn(batch, n, K, generator=g, device="cuda") / K**0.5).to(BF16)
    bias = torch.randn(n, generator=g, device="cuda") if epi < 2 else None
    out = torch.full((R + 1, width + 8), 7.0, dtype=odt, device="cuda")
    common = dict(batch=batch, lda=K + 8, sbn=K, b_bs=n * K, epi=epi, limit=0.75, bias=bias, n_out=width if epi >= 2 else 0)
    if lens:
        offs = torch.tensor([sum(lens[:i]) for i in range(batch + 1)], dtype=torch.int32, device="cuda")
        perm = torch.randperm(R, generator=g, device="cuda").to(torch.int32)
        scale = torch.rand(R, generator=g, device="cuda") + 0.5
        S.bgemm(a, w, out, R, n, K, grp_offs=offs, a_rows=perm, a_div=2, c_rows=perm, row_scale=scale, **common)
        groups = [(perm[int(offs[b]) : int(offs[b + 1])].long() // 2, perm[int(offs[b]) : int(offs[b + 1])].long()) for b in range(batch)]
    else:
        S.bgemm(a, w, out, each, n, K, a_bs=each * (K + 8), c_bs=each * (width + 8), **common)
        scale = torch.ones(R, device="cuda")
        groups = [(torch.arange(b * each, (b + 1) * each, device="cuda"),) * 2 for b in range(batch)]
    assert bool((out[R:] == 7).all()) and bool((out[:, width:] == 7).all())  # nothing beyond the rows and columns
    # a sum of K products of about 1 / sqrt(K) in fp32 is off by 2^-24 sqrt(K) of its size at most, squared and gated twice that, the epilogue's few operations 2^-22; a bf16 result (eight significant bits) by 2^-8
    tol = 2**-24 * (2 * K**0.5 + 8) + (2**-8 if odt == BF16 else 0.0)
    for b, (src, dst) in enumerate(groups):
        if not len(src):
            continue
        y = a[src].double() @ w[b].double().mT
        if epi >= 2:
            v = y.view(len(src), -1, 2, 32)
            gt, up = (v[:, :, i].flatten(1)[:, :width] for i in (0, 1))
            if epi == 2:
                y = gt.clamp(max=0.75) * torch.sigmoid(1.702 * gt.clamp(max=0.75)) * (up.clamp(-0.75, 0.75) + 1)
            else:
                y = (torch.nn.functional.silu(gt) if epi == 4 else torch.nn.functional.gelu(gt, approximate="tanh")) * up
        else:
            y = y + bias.double()
            y = torch.relu(y) ** 2 if epi == 1 else y
        y = y * scale[dst].double()[:, None]
        got = out[dst, :width].double()
        rows = (got - y).norm(dim=1) / (y.norm(dim=1) + 1e-30)  # row by row: one that came from another place is off by about its size
        assert float(rows.max()) < tol, (b, len(src))


@pytest.mark.parametrize("K,epi,quad", [(640, 0, False), (768, 0, True), (640, 1, False), (768, 1, True), (384, 4, False), (512, 4, True), (1152, 2, False), (1280, 2, True), (1152, 3, False), (1280, 3, True), (832, 0, False)])
def test_which_sums_of_groups_take_four_waves(K, epi, quad):
    a, w, out = torch.zeros(900, K, dtype=BF16, device="cuda"), torch.zeros(8, 2048, K, dtype=BF16, device="cuda"), torch.empty(900, 1024 if epi >= 2 else 2048, dtype=BF16, device="cuda")
    offs = torch.tensor([0, 100, 100, 300, 440, 460, 700, 899, 900], dtype=torch.int32, device="cuda")

    def run():
        S.bgemm(a, w, out, 900, 2048, K, grp_offs=offs, batch=8, lda=K, sbn=K, b_bs=2048 * K, epi=epi, limit=1.0, n_out=1024 if epi >= 2 else 0)
        torch.cuda.synchronize()

    run()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as p:
        run()
    assert any("bgemm_quad_kernel" in e.key for e in p.key_averages()) is quad
