"""Chunks whose tiles of 64 x 64 and 64 x 128 are computed by four waves that share the contraction: numbers of stages below, at
and beyond the ring of four, ragged tiles in both directions, at the edges of each kernel's range, and rotation tables at any alignment."""

import pytest
import torch

from test_gpu_append import make_layer, rope_tables, test_prefill_chunks_take_the_large_tiles as check_chunk
from tpa import tpa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("paged", [False, True])
@pytest.mark.parametrize(
    "b,n,dm,h,d,rq,rk",
    [
        (3, 71, 64, 64, 64, 16, 8),      # 64 x 64: one stage, 4 x 64 tiles
        (1, 257, 128, 16, 128, 6, 2),    # two; one token in the last tile, 32 columns
        (2, 90, 192, 32, 128, 6, 2),     # three
        (1, 200, 256, 32, 128, 6, 2),    # four
        (4, 60, 320, 8, 64, 6, 2),       # five; 720 columns
        (1, 129, 704, 24, 96, 5, 3),     # eleven; 1320 columns, no power of two anywhere
        (1, 300, 4096, 32, 128, 6, 2),   # 64
        (1, 1100, 1984, 8, 64, 6, 2),    # 18 x 12 tiles
        (9, 100, 1984, 32, 128, 6, 2),   # 15 x 25 tiles, below the range of the next
        (1, 693, 2048, 32, 128, 6, 2),   # 64 x 128: 11 x 13 tiles, a half in the last column
        (2, 1200, 2112, 8, 64, 6, 2),    # 33 stages; 38 x 6 tiles
        (1, 520, 2048, 64, 64, 16, 4),   # 9 x 24 tiles, eight tokens in the last
        (1, 2433, 2048, 8, 96, 5, 2),    # 39 x 15 = 585: beyond
    ],
)
def test_waves_share_the_contraction(gpu, b, n, dm, h, d, rq, rk, paged):
    check_chunk(gpu, b, n, dm, h, d, rq, rk, paged)


@pytest.mark.parametrize("n,dm", [(150, 256), (700, 2048), (2700, 128)])  # the last: 128 x 128 tiles where the tables are aligned, 64 x 64 else
def test_tables_at_any_alignment(gpu, n, dm):
    h, d, rq, rk = 8, 64, 6, 2
    x, w = make_layer(21, 1, n, dm, h, d, rq, rk, torch.bfloat16, gpu)
    tables = [torch.from_numpy(t).to(gpu) for t in rope_tables(n + 8, d)]
    outs = []
    for shift in (0, 1, 3):
        cos, sin = (torch.cat([t.new_zeros(shift), t.flatten()])[shift:].view(t.shape) for t in tables)
        caches = [torch.zeros((1, n, rk, inner), dtype=torch.bfloat16, device=gpu) for inner in (h, d, h, d)]
        qa, qb, _ = tpa.tpa_cache_append(x, w, cos, sin, *caches, rank_q=rq, kernel=2)
        outs.append([qa, qb] + caches)
    for got in outs[1:]:
        for a, b in zip(outs[0], got):
            # another order of the same fp32 sums at most, each rounded once to 8 bits
            assert (a.float() - b.float()).abs().max() <= 2.0**-8 * a.float().abs().max()
            assert n > 2000 or torch.equal(a, b)
