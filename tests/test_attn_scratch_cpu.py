"""The scratch of the attention backward, without a GPU: what is kept between calls when memory is short."""
import weakref

import pytest
import torch

from llm_quest_amd import kernels as K


@pytest.fixture
def memory(monkeypatch):
    """A device with "free" bytes, whose allocations are counted ("made") and, once dropped, cached."""
    state, live, real = {"free": 0, "made": [], "top": 0}, [], torch.empty

    def empty(n, **kw):
        state["made"].append(n)
        state["free"] -= max(0, n - cached())
        t = real(n, dtype=torch.uint8)
        live.append(weakref.ref(t))
        state["top"] = max(state["top"], allocated())
        return t

    def allocated(device=None):
        return sum(t().numel() for t in live if t() is not None)

    def cached():
        return state["top"] - allocated()

    monkeypatch.setattr(K, "_ATTN_WS", {})
    monkeypatch.setattr(K.L, "stream", lambda device: 7)
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda device: (state["free"], 0))
    monkeypatch.setattr(torch.cuda, "memory_reserved", lambda device: state["top"])
    monkeypatch.setattr(torch.cuda, "memory_allocated", allocated)
    monkeypatch.setattr(torch, "empty", empty)
    return state


def test_a_buffer_stays_where_a_larger_one_is_not_granted(memory, monkeypatch):
    monkeypatch.setattr(K.L, "load", lambda: type("lib", (), {"mi355_attn_bwd_split_bytes": staticmethod(lambda *a: 600)}))
    dev = torch.device("cuda", 0)
    memory["free"] = 4400  # a quarter: 1 100, room for the scratch of 1 000 and not for the parts behind it
    for _ in range(3):
        ws, size = K._attn_split_scratch(dev, 1000, 1, 2, 1, 1, 128, True)
        assert size == 1000 and ws.numel() == 1000 and memory["made"] == [1000]
        del ws
    memory["free"] = 6000  # and the 1 000 that it would give back: a quarter is 1 750
    ws, size = K._attn_split_scratch(dev, 1000, 1, 2, 1, 1, 128, True)
    assert size == 1600 and memory["made"] == [1000, 1600] and [t.numel() for t in K._ATTN_WS.values()] == [1600]


def test_what_is_not_granted_takes_nothing_away(memory):
    dev = torch.device("cuda", 0)
    memory["free"] = 4000
    assert K._attn_scratch(dev, 900).numel() == 900
    memory["free"] = 0
    assert K._attn_scratch(dev, 5000) is None and K._attn_scratch(dev, 900).numel() == 900 and memory["made"] == [900]


@pytest.mark.parametrize("B,S,Hq,Hkv,causal,cut", [
    (128, 1, 4, 1, True, False), (128, 17, 4, 1, False, False), (8, 65, 16, 8, True, False), (2, 197, 16, 16, False, False), (3, 256, 16, 16, False, False), (8, 257, 4, 4, False, False),
    (8, 256, 16, 8, False, False), (8, 129, 16, 8, False, False), (1, 128, 16, 8, True, True), (1, 300, 16, 8, True, True), (2, 498, 16, 8, True, True), (1, 709, 16, 8, True, True), (3, 560, 16, 8, True, True),
    (1, 1500, 16, 8, True, True), (1, 2000, 16, 8, False, True), (2, 257, 16, 16, True, True), (8, 256, 16, 8, True, True), (32, 64, 4, 1, True, True), (2, 498, 16, 16, True, True), (7, 584, 4, 4, True, True)])
def test_which_key_blocks_are_split(B, S, Hq, Hkv, causal, cut):
    """Split where the longest chain of tiles becomes shorter by more than the parts cost to write and add up, whole where it does not (both sides measured)."""
    assert (K.L.load().mi355_attn_bwd_split_bytes(B, S, Hq, Hkv, 128, int(causal)) > 0) is cut
