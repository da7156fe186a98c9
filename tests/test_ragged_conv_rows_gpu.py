"""Causal convolution of long packed steps (eight rows to a thread): sequences that start, end and lie wholly inside the eight, old state, every kind of row -- against the rows one sequence at a time."""
import pytest
import torch

pytestmark = pytest.mark.gpu
F32 = torch.float32


@pytest.mark.parametrize("C,taps", [(1028, 2), (1028, 3), (1028, 4), (1028, 8), (4100, 2), (4100, 3), (300, 4), (768, 4)])  # (4 200 x 1 028 rows of two taps, and of three in bf16, stay with a row a thread)
@pytest.mark.parametrize("sizes", [(4097,), (1, 1, 1, 4200), (2049, 3, 8, 5, 1, 2100), (7,) * 600])
@pytest.mark.parametrize("dtype,act,residual", [(torch.bfloat16, True, False), (F32, False, True)])
def test_packed_rows_are_the_sequences_one_by_one(C, taps, sizes, dtype, act, residual):
    from llm_quest_amd import kernels_seq as S

    n = len(sizes)
    T = sum(sizes)
    g = torch.Generator(device="cuda").manual_seed(T + taps)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    x = torch.randn(T, C, generator=g, device="cuda").to(dtype)
    w, bias = torch.randn(C, taps, generator=g, device="cuda"), torch.randn(C, generator=g, device="cuda")
    state = torch.randn(n + 2, taps - 1, C, generator=g, device="cuda")
    alone = state.clone()
    off = [0, *torch.tensor(sizes).cumsum(0).tolist()]
    rows = torch.repeat_interleave(torch.arange(n), torch.tensor(sizes)).to(torch.int32).cuda()
    slot = torch.randperm(n + 2, generator=torch.Generator().manual_seed(T))[:n].to(torch.int32).cuda()
    got = S.ragged_conv(x, w, state, rows, i32(off), slot, act=act, residual=residual, out_dtype=F32, bias=bias)
    padded = torch.cat([torch.cat([alone[int(slot[i])].double(), x[off[i] : off[i + 1]].double()]) for i in range(n)])
    want = torch.empty(T, C, dtype=torch.float64, device="cuda")
    for i in range(n):
        part = padded[off[i] + i * (taps - 1) : off[i + 1] + (i + 1) * (taps - 1)]
        want[off[i] : off[i + 1]] = bias.double() + sum(w[:, j].double() * part[j : j + sizes[i]] for j in range(taps))
        assert torch.equal(state[int(slot[i])], part[-(taps - 1) :].float())
    want = (torch.nn.functional.silu(want) if act else want) + (x.double() if residual else 0)
    # taps + 2 fp32 roundings of numbers below about 20, then an exponential and a quotient of one or two units each
    assert float((got.double() - want).abs().max()) < 2e-5
    if n < 10:  # the same bits as the kernel of short steps
        for i in range(n):
            lo = max(off[i], off[i + 1] - 3)
            st = torch.cat([alone[int(slot[i])], x[off[i] : off[i + 1]].float()])[lo - off[i] : lo - off[i] + taps - 1][None].contiguous()
            k = off[i + 1] - lo
            few = S.ragged_conv(x[lo : off[i + 1]].contiguous(), w, st, i32([0] * k), i32([0, k]), i32([0]), act=act, residual=residual, out_dtype=F32, bias=bias)
            assert torch.equal(few, got[lo : off[i + 1]])
