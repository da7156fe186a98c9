"""Which input gradients are worth a transposed copy of their weight."""
import pytest

from llm_quest_amd.kernels import dgrad_on_quad, dgrad_transposes


@pytest.mark.parametrize("M,N,K,copies", [
    (1416, 1024, 4096, True), (1280, 1024, 4096, True), (1279, 1024, 4096, False), (1280, 4096, 8192, True), (1280, 4097, 8192, False),  # rows; outputs up to half of the sums
    (1280, 1024, 2048, False), (1900, 1024, 2048, False), (1910, 1024, 2048, True), (2836, 64, 8192, False), (1280, 512, 8192, True), (1700, 256, 8192, False),  # enough work for the copy
    (1280, 1024, 16320, True), (1999, 1024, 16328, False), (2000, 1024, 16328, True), (1280, 4096, 16384, False), (2836, 4096, 16384, True), (4095, 1024, 16392, False),  # sums that the NN form divides
    (4095, 1024, 248320, False), (1340, 8160, 16320, True), (4096, 64, 64, True), (17016, 1024, 151936, True), (2000, 2047, 2040, False)])
def test_where_the_lines_lie(M, N, K, copies):
    assert dgrad_transposes(M, N, K) is copies


@pytest.mark.parametrize("M,N,K,epilogue,quad", [
    (33_000, 3072, 256, False, False), (33_000, 3072, 320, False, False), (33_000, 3072, 576, False, False), (33_000, 3072, 512, False, True), (33_000, 3072, 704, False, True),  # short sums over two rounds of tiles
    (33_000, 3072, 320, True, True), (33_000, 3072, 192, True, False), (16_000, 2048, 320, False, True), (16_384, 2048, 320, False, False),  # behind SwiGLU; 504 and 512 tiles
    (4096, 2048, 1024, False, False), (4352, 2048, 1024, False, True), (300, 256, 16_384, False, False), (300, 256, 16_448, False, True), (300, 256, 16_448, True, False), (8192, 2052, 1024, False, False), (8192, 2048, 1000, False, False)])
def test_which_take_the_weight_as_it_lies(M, N, K, epilogue, quad):
    assert dgrad_on_quad(M, N, K, epilogue=epilogue) is quad
