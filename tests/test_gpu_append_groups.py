"""Chunks whose 128 x 128 tiles are computed by two groups of waves, each half of the contraction: numbers of k steps per
group that end in either register set, and more sequences than a group has threads."""

import pytest

from test_gpu_append import test_prefill_chunks_take_the_large_tiles as check_chunk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(
    "b,n,dm",
    [
        (3, 700, 256),   # two steps per group
        (3, 700, 384),   # three
        (2, 1025, 512),  # four, ragged last tile of tokens
        (300, 7, 640),   # five; 300 sequences
        (3, 700, 320),   # an odd number of steps in all: one group
    ],
)
@pytest.mark.parametrize("paged", [False, True])
def test_two_groups_share_the_contraction(gpu, b, n, dm, paged):
    check_chunk(gpu, b, n, dm, 16, 128, 6, 2, paged)
