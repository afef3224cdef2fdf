"""The append kernel for few tokens (16 columns and up to 64 tokens per workgroup, the contraction in eight parts, one to a wave, in
chunks of 64): numbers of tokens around its blocks of 16, 32 and 64, contractions of fewer chunks than waves and of odd
numbers of chunks, ragged column blocks, and calls on either side of the line to the 64 x 64 tiles, against the CPU oracle."""

import pytest
import torch

from tpa import tpa

from test_gpu_append import test_append_matches_the_oracle as check_append

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(
    "b,n,dm,h,d,rq,rk",
    [
        (1, 1, 4096, 32, 128, 6, 2),   # blocks of 16 tokens, 15 of them past the end
        (17, 1, 192, 8, 64, 2, 1),     # three chunks of k: five waves have none; a second block of one token
        (11, 3, 1088, 32, 128, 6, 2),  # 17 chunks; 33 tokens x 100 column blocks: blocks of 32
        (13, 5, 64, 32, 128, 6, 2),    # one chunk of k: seven waves have none
        (13, 5, 1024, 32, 128, 6, 2),  # 65 tokens: two blocks of 64, the last of one token
        (1, 20, 576, 64, 64, 16, 8),   # 256 column blocks, nine chunks: one wave has two; blocks of 32
        (3, 5, 2048, 32, 128, 16, 8),  # 15 tokens x 320 column blocks, two rounds of blocks of 16
        (3, 30, 2112, 8, 64, 1, 1),    # 33 chunks; 216 columns: the last block owns 8 of its 16
        (2, 83, 512, 64, 64, 16, 8),   # 166 tokens x 256 column blocks, 768 workgroups: tiles
        (3, 71, 512, 64, 64, 16, 8),   # 213 tokens, 1024: tiles
        (4, 63, 512, 32, 128, 6, 2),   # 252 tokens x 100 column blocks, two rounds of blocks of 64 tokens: tiles
        (4, 63, 4096, 32, 128, 6, 2),  # the same, 64 chunks
    ],
)
def test_append_few_tokens(gpu, b, n, dm, h, d, rq, rk):
    check_append(gpu, torch.bfloat16, 2, b, n, dm, h, d, rq, rk, False)


@pytest.mark.parametrize(
    "b,n,dm,h,d,rq,rk",
    [
        (2, 75, 5120, 16, 128, 6, 2),  # two rounds of blocks of 32: from here on they are the faster side
        (2, 75, 5056, 16, 128, 6, 2),  # and below tiles of 64 x 64
        (2, 80, 4096, 8, 64, 6, 2),    # one round
        (3, 64, 5120, 32, 128, 6, 2),  # three rounds: tiles
    ],
)
def test_append_at_the_line_to_the_tiles(gpu, b, n, dm, h, d, rq, rk):
    check_append(gpu, torch.bfloat16, 2, b, n, dm, h, d, rq, rk, False)


def test_results_are_the_roundings_of_exact_sums(gpu):
    """Results of a long contraction that are not the bf16 rounding of the exact sum.  An fp32 sum that is off by e rounds to the
    wrong side for a share of about 2 e / spacing of the results; with the chunks of 64 summed one by one that is 1.7e-4 here, with one
    chain of matrix instructions per wave 3.2e-4 (1.8 million results: 310 and 590, give or take 25)."""
    n, dm, h, d, rq, rk = 48, 16384, 32, 128, 6, 2
    wrong = total = 0
    for seed in range(24):
        g = torch.Generator(device="cuda").manual_seed(seed)
        x = torch.randn((1, n, dm), generator=g, device=gpu).to(torch.bfloat16)
        w = (torch.randn(((rq + 2 * rk) * (h + d), dm), generator=g, device=gpu) * dm**-0.5).to(torch.bfloat16)
        cos, sin = torch.ones((n, d // 2), device=gpu), torch.zeros((n, d // 2), device=gpu)
        kv = [torch.zeros((1, n, rk, e), dtype=torch.bfloat16, device=gpu) for e in (h, d, h, d)]
        qa, qb, _ = tpa.tpa_cache_append(x, w, cos, sin, *kv, torch.zeros(1, dtype=torch.int32, device=gpu), rank_q=rq, kernel=2)
        got = torch.cat([t.reshape(n, -1) for t in (qa, qb, *kv)], dim=1)
        want = (x[0].double() @ w.double().T).float().to(torch.bfloat16)
        wrong += int((got != want).sum())
        total += got.numel()
    assert wrong <= 2.4e-4 * total, wrong / total
