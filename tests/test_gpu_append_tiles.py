"""Appends between a decode step and a large chunk: the 64 x 64 tiles with their contraction dealt to one, two or four groups of
waves, the lines to the kernels on either side, and the order in which the tiles are dealt out, against the CPU oracle."""

import pytest

from test_gpu_append import test_prefill_chunks_take_the_large_tiles as check_chunk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("paged", [False, True])
@pytest.mark.parametrize(
    "b,n,dm,h,d,rq,rk",
    [
        (2, 50, 512, 64, 64, 16, 8),   # 512 workgroups of the few-token kernel: four groups; 2 x 64 tiles, columns outside
        (3, 71, 64, 64, 64, 16, 8),    # one step: three groups have none; ragged last tile of tokens
        (1, 256, 320, 64, 64, 16, 8),  # 256 tiles, the most for four groups; five steps: the first group has two
        (1, 257, 192, 64, 64, 16, 8),  # 320: two groups, three steps
        (5, 120, 448, 8, 64, 6, 2),    # 720 columns: the last tile owns 16; 10 x 12 tiles
        (1, 1100, 128, 8, 64, 6, 2),   # 18 x 12 tiles, tokens outside
        (4, 128, 128, 64, 64, 16, 8),  # 512 tiles, the most for two groups
        (1, 513, 128, 64, 64, 16, 8),  # 576: 128 x 128 tiles, 5 x 32 of them
        (2, 1216, 64, 64, 64, 16, 8),  # 19 x 32 tiles of 128 x 128
        (1, 2433, 64, 64, 64, 16, 8),  # 20 x 32
    ],
)
def test_append_of_chunks_of_all_sizes(gpu, b, n, dm, h, d, rq, rk, paged):
    check_chunk(gpu, b, n, dm, h, d, rq, rk, paged)


@pytest.mark.parametrize(
    "b,n,dm,h,d,rq,rk",
    [
        (1, 2433, 2112, 64, 64, 16, 8),  # 20 x 32 tiles, three per compute unit, above 2048: 10 x 16 tiles of 256 x 256
        (1, 2433, 2048, 64, 64, 16, 8),  # 2048: they stay
        (3, 2731, 1024, 32, 128, 6, 2),  # 65 x 13, four: 33 x 7 tiles of 256 x 256, one token in the last and 64 columns
        (5, 2000, 1088, 16, 128, 7, 1),  # 79 x 11: rank rows and factors change inside a wave's 64-column pieces
    ],
)
def test_append_of_large_chunks(gpu, b, n, dm, h, d, rq, rk):
    check_chunk(gpu, b, n, dm, h, d, rq, rk, False)
