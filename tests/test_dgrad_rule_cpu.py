"""Which input gradients are worth a transposed copy of their weight."""
import pytest

from llm_quest_amd.kernels import dgrad_transposes


@pytest.mark.parametrize("M,N,K,copies", [
    (1416, 1024, 4096, True), (1280, 1024, 4096, True), (1279, 1024, 4096, False), (1280, 4096, 8192, True), (1280, 4097, 8192, False),  # rows; outputs up to half of the sums
    (1280, 1024, 2048, False), (1900, 1024, 2048, False), (1910, 1024, 2048, True), (2836, 64, 8192, False), (1280, 512, 8192, True), (1700, 256, 8192, False),  # enough work for the copy
    (1280, 1024, 16320, True), (1999, 1024, 16328, False), (2000, 1024, 16328, True), (1280, 4096, 16384, False), (2836, 4096, 16384, True), (4095, 1024, 16392, False),  # sums that the NN form divides
    (4095, 1024, 248320, False), (1340, 8160, 16320, True), (4096, 64, 64, True), (17016, 1024, 151936, True), (2000, 2047, 2040, False)])
def test_where_the_lines_lie(M, N, K, copies):
    assert dgrad_transposes(M, N, K) is copies
