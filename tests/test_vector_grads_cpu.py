"""What a block's backward hands over to be added up (``kernels.reduce_rows_each``), with every kernel replaced by plain arithmetic: the sums of one launch have no order, so none of them may meet another's
destination, and every parameter gets the sum of all its contributions, parameters that a block holds twice too."""

from types import SimpleNamespace

import pytest
import torch

from llm_quest_amd import _lib as L
from llm_quest_amd import ops, ops_q35
from llm_quest_amd.qwen.qwen3.qwen3_transformer_block import TransformerBlock
from llm_quest_amd.qwen.qwen3_5.qwen3_5_text_model import Qwen3_5TransformerBlock

BF16, F32 = torch.bfloat16, torch.float32
D, HEAD = 16, 8


class Kernels:
    """Stands in for kernels.py and kernels_q35.py: rows to be added up are whole numbers, so a sum has one value; everything else is a matrix of no interest."""

    def __init__(self):
        self.g, self.given, self.launches, self.fails = torch.Generator().manual_seed(3), [], 0, None

    def __getattr__(self, name):
        def call(*a, **kw):
            return torch.zeros(4, D, dtype=BF16)

        return call

    def rows(self, n):
        if len(self.given) == self.fails:
            raise MemoryError
        self.given.append(torch.randint(-4, 5, (3, n), generator=self.g).float())
        return self.given[-1]

    def rmsnorm_bwd(self, x, w, rstd, dy, dres=None, partial=False):
        return torch.zeros(4, D, dtype=BF16), self.rows(D)

    def dgrad_attn_delta(self, *a):
        return None

    def attn_bwd_qnorm(self, *a, **kw):
        return self.rows(HEAD)

    def qknorm_rope_bwd(self, *a, **kw):
        return None, self.rows(HEAD)

    def headnorm_rope_bwd(self, *a, **kw):
        return self.rows(HEAD)

    def gated_rmsnorm_bwd(self, *a, **kw):
        return torch.zeros(4, 2 * HEAD, dtype=BF16), self.rows(HEAD)

    def causal_conv_silu_bwd(self, x, w, *a, **kw):
        return self.rows(w.numel())

    def gdn_gates_bwd(self, b, a, log_A, *rest, **kw):
        return self.rows(log_A.numel()), self.rows(log_A.numel())

    def gated_delta_rule_bwd(self, *a, **kw):
        return (None,) * 4

    def reduce_rows_each(self, sums):
        assert 1 <= len(sums) <= 4
        self.launches += 1
        spans = sorted((out.data_ptr(), out.data_ptr() + out.numel() * out.element_size()) for _, out, _ in sums)
        assert all(a[1] <= b[0] for a, b in zip(spans, spans[1:])), "two sums of one launch have the same destination"
        for part, out, acc in reversed(sums):  # (in no order)
            total = part.sum(0).view(out.shape)
            out.copy_(out.float() + total if acc else total)


@pytest.fixture
def kernels(monkeypatch):
    k = Kernels()
    for m, names in ((ops, ("K",)), (ops_q35, ("K", "Q"))):
        for n in names:
            monkeypatch.setattr(m, n, k)
    return k


def qwen3():
    blk = TransformerBlock(dict(emb_dim=D, hidden_dim=32, n_heads=2, num_kv_groups=1, head_dim=HEAD, dtype=BF16), 0)
    m = torch.zeros(4, 4 * HEAD, dtype=BF16)
    saved = (None, None, None, m, (m, m[:, : 2 * HEAD], m[:, :HEAD], None, None), None, None, None, None, None)
    rt = SimpleNamespace(B=1, S=4, cos=None, sin=None, pos=None, key_mask=None)
    return blk, lambda: ops.block_backward(blk, saved, torch.zeros(4, D, dtype=BF16), rt)


def hybrid(layer):
    blk = Qwen3_5TransformerBlock(dict(emb_dim=D, hidden_dim=32, n_heads=2, num_kv_groups=1, head_dim=HEAD, dtype=BF16, linear_num_qk_heads=2, linear_num_value_heads=2, linear_qk_head_dim=HEAD,
                                       linear_value_head_dim=HEAD, linear_conv_kernel_size=4, linear_sdpa_ratio=4, mrope_section=None, partial_rope_factor=0.25, p_dropout=0.0, training=False), layer)
    m = torch.zeros(4, 16 * HEAD, dtype=BF16)
    mixer = (m,) * 10 if blk.is_linear else (m,) * 9 + (None,)
    saved = (None, None, m, None, m, mixer, None, None, None, None, None, None)
    rt = SimpleNamespace(B=1, S=4, cos_t=None, sin_t=None, pos=None, key_mask=None)
    return blk, lambda: ops_q35.block_backward(blk, saved, torch.zeros(4, D, dtype=BF16), rt)


# (the block, which of its parameters are which others, the parameters in the order that the backward reaches them)
QWEN3 = ["norm2.weight", "att.q_norm.weight", "att.k_norm.weight", "norm1.weight"]
DELTA = ["norm2.scale", "att.post_norm.weight", "att.conv1d.weight", "att.log_A", "att.dt_bias", "norm1.scale"]
GATED = ["norm2.scale", "att.q_norm.scale", "att.k_norm.scale", "norm1.scale"]
CASES = [(qwen3, QWEN3, {}), (qwen3, QWEN3, {"att.k_norm": "att.q_norm"}), (qwen3, QWEN3, {"norm2": "norm1", "att.k_norm": "att.q_norm"}), (lambda: hybrid(3), GATED, {"att.k_norm": "att.q_norm"}),
         (lambda: hybrid(0), DELTA, {}), (lambda: hybrid(0), DELTA, {"norm2": "norm1"})]


@pytest.mark.parametrize("make,order,tied", CASES)
def test_every_vector_gradient_is_the_sum_of_its_contributions(kernels, make, order, tied):
    blk, backward = make()
    for a, b in tied.items():
        (owner, name), (other, theirs) = a.rpartition(".")[::2], b.rpartition(".")[::2]
        setattr(blk.get_submodule(owner), name, getattr(blk.get_submodule(other), theirs))
    params = [blk.get_parameter(n) for n in order]
    want = {}
    for _ in range(2):  # a second pass adds to the first one's
        kernels.given.clear()
        backward()
        for p, part in zip(params, kernels.given):
            want[p] = want.get(p, 0) + part.sum(0).view(p.shape)
        assert len(kernels.given) == len(params)
    for p, total in want.items():
        assert p.grad.dtype == p.dtype and torch.equal(p.grad.float(), total)
    if not tied:
        assert kernels.launches == 2 * ((len(order) + 3) // 4)


@pytest.mark.parametrize("make,order", [(qwen3, QWEN3), (lambda: hybrid(3), GATED), (lambda: hybrid(0), DELTA)])
def test_a_backward_that_ends_early_leaves_no_unwritten_gradient(kernels, make, order):
    """An allocation fails in front of one of the sums: the gradients are what they were, none at first and then the first pass's, and the pass that follows adds to those."""
    blk, backward = make()
    params, want = [blk.get_parameter(n) for n in order], None
    for _ in range(2):
        for fails in range(len(order)):
            kernels.given.clear()
            kernels.fails = fails
            with pytest.raises(MemoryError):
                backward()
            assert all(p.grad is None for p in params) if want is None else all(torch.equal(p.grad.float(), t) for p, t in zip(params, want))
        kernels.given.clear()
        kernels.fails = None
        backward()
        want = [part.sum(0).view(p.shape) + (0 if want is None else want[i]) for i, (p, part) in enumerate(zip(params, kernels.given))]
        assert all(torch.equal(p.grad.float(), t) for p, t in zip(params, want))


def test_fp32_gradients_in_one_tensors_memory(kernels):
    """A program may have given stand-alone parameters gradients that share memory: both sums arrive, as one launch behind the other."""
    blk, backward = hybrid(0)
    a, b = blk.att.post_norm.weight, blk.att.log_A
    memory = torch.zeros(HEAD)
    a.grad, b.grad = memory, memory[1:3]
    backward()
    want = kernels.given[1].sum(0)
    want[1:3] += kernels.given[3].sum(0)
    assert torch.equal(memory, want)


@pytest.mark.parametrize("tied", [{}, {"ffn.lin2": "att.out_proj"}, {"att.out_proj": "att.w_keys"}, {"ffn.lin2": "att.w_queries", "att.out_proj": "att.w_values"}])
def test_a_weight_that_a_block_holds_twice_is_in_one_grouped_launch_once(kernels, tied, monkeypatch):
    """The products of a grouped launch have no order either."""
    blk = TransformerBlock(dict(emb_dim=D, hidden_dim=D, n_heads=2, num_kv_groups=2, head_dim=HEAD, dtype=BF16), 0)
    for a, b in tied.items():
        (owner, name), (other, theirs) = a.rpartition(".")[::2], b.rpartition(".")[::2]
        setattr(blk.get_submodule(owner), name, getattr(blk.get_submodule(other), theirs))
    arena, g, want, wg = ops.arena_for(blk), torch.Generator().manual_seed(5), {}, []
    att, ffn = blk.att, blk.ffn
    launched = []

    def gemm_grouped(form, problems):
        spans = sorted((out.data_ptr(), out.data_ptr() + out.numel() * out.element_size()) for _, _, out, _ in problems)
        assert all(a[1] <= b[0] for a, b in zip(spans, spans[1:])), "two products of one launch have the same destination"
        launched.append(len(problems))
        for dy, x, out, r in reversed(problems):
            out.copy_(dy.float().T @ x.float() + (0 if r is None else r.float()))

    monkeypatch.setattr(kernels, "gemm_grouped", gemm_grouped, raising=False)
    for _ in range(2):
        for first, last, rows in ((ffn.lin2, None, D), (ffn.lin1, ffn.lin_gate, 2 * D), (att.out_proj, None, D), (att.w_queries, att.w_values, 6 * HEAD)):
            dy, x = (torch.randint(-2, 3, (4, n), generator=g).to(BF16) for n in (rows, D))
            ops._wgrad(arena, first.weight, None if last is None else last.weight, dy, x, wg)
            total = dy.float().T @ x.float()
            parts = [first] if last is None else [ffn.lin1, ffn.lin_gate] if first is ffn.lin1 else [att.w_queries, att.w_keys, att.w_values]
            for m, t in zip(parts, total.split([m.weight.shape[0] for m in parts])):
                want[m.weight] = want.get(m.weight, 0) + t
        ops._flush_wgrads(wg)
        assert not wg
    assert all(torch.equal(p.grad.float(), t) for p, t in want.items())
    assert tied or launched == [4, 4]


def test_overlapping_destinations_are_refused():
    """By the entry point itself, before anything is launched."""
    part, out = torch.zeros(2, 8), torch.zeros(24)
    at = lambda i, n, dt=0: (part.data_ptr(), 8, 2, n, out.data_ptr() + 4 * i, dt)
    none = (None, 0, 0, 0, None, 0)
    for sums in ([at(0, 8), at(0, 8)], [at(0, 8), none, at(7, 8)], [at(8, 8), at(16, 8), at(4, 8)], [at(0, 8, 1), at(3, 8, 1)], [none, at(8, 8), none, at(11, 8, 3)]):
        sums = sums + [none] * (4 - len(sums))
        assert L.load().mi355_reduce_rows_each(*[x for s in sums for x in s], None) != 0
        assert "overlaps" in L.load().mi355_last_error().decode()
