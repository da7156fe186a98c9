"""How many workgroups share a head's keys in a one-token step."""
import pytest

from llm_quest_amd.ops_decode import decode_splits, step_splits


@pytest.mark.parametrize("n_keys,splits", [(1, 1), (256, 1), (257, 3), (596, 5), (1024, 8), (1025, 8), (2028, 8), (4064, 8), (8192, 8), (9216, 9), (12288, 12), (32128, 12), (1 << 20, 12)])
def test_one_sequence_is_folded_from_few_splits(n_keys, splits):
    """Splits that the output projection folds: 128 keys each up to eight, then eight until a split has 1 024 keys, at most twelve."""
    assert step_splits(n_keys, 1, 16) == splits


def test_never_more_workgroups_than_there_are_units():
    for heads in (1, 4, 16, 40, 64, 128, 300):
        for n in (1, 300, 5000, 100000):
            assert 1 <= step_splits(n, 1, heads) <= max(1, 256 // heads)
            assert all(step_splits(n, B, heads) == decode_splits(n, B, heads) for B in (2, 5, 8))
