"""Batch entries of different lengths, which start longest first and share every XCD: each entry's rows are what a call of that entry
alone gives, whatever the lengths, the blocks, the ranges of keys and the mask."""

import pytest
import torch


@pytest.mark.gpu
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize(
    "b,h,d,lq,lk,rk,lengths",
    [
        (4, 48, 64, 300, 700, 2, [300, 64, 700, 600]),             # too short to be ordered
        (3, 64, 128, 300, 700, 2, [0, 700, 1]),
        (7, 32, 128, 260, 900, 2, [800, 900, 790, 900, 900, 800, 801]),
        (5, 32, 64, 513, 1100, 2, [300, 1100, 300, 900, 1100]),
        (6, 40, 128, 260, 600, 4, [65, 600, 300, 0, 600, 1]),
        (6, 32, 128, 300, 4000, 2, [1500, 4000, 64, 0, 3000, 3001]),  # the fewest workgroups, the keys in ranges
        (64, 8, 64, 17, 200, 2, [3 * i + 1 for i in range(64)]),
        (65, 8, 64, 17, 200, 8, [3 * i + 1 for i in range(65)]),
        (4, 48, 64, 300, 2047, 2, [300, 64, 2047, 1600]),          # one key below the line, and at it
        (4, 48, 64, 300, 2048, 2, [300, 64, 2048, 1600]),
        (3, 64, 128, 300, 2100, 2, [0, 2100, 1]),                  # no key, one key
        (7, 32, 128, 260, 2200, 2, [2000, 2200, 1990, 2200, 2200, 2000, 2001]),  # alike: the order of equal lengths
        (5, 32, 64, 513, 2300, 2, [300, 2300, 300, 1900, 2300]),   # equal ones among them, three blocks
        (6, 40, 128, 260, 2600, 4, [65, 2600, 300, 0, 2600, 1]),   # dense tiles
        (7, 64, 64, 260, 2500, 8, [65, 2500, 300, 0, 2500, 1, 64]),
        (32, 16, 64, 17, 2100, 2, [65 * i + 1 for i in range(32)]),  # as many as are ordered
        (33, 16, 64, 17, 2100, 2, [65 * i + 1 for i in range(33)]),  # and one more
    ],
)
def test_entries_are_what_they_are_alone(gpu, b, h, d, lq, lk, rk, lengths, causal):
    from tpa import tpa

    gen = torch.Generator(device=gpu).manual_seed(lq + lk)
    make = lambda l, r, x: (torch.randn((b, l, r, x), generator=gen, device=gpu) / r**0.5).to(torch.bfloat16)
    args = [make(l, r, x) for l, r in ((lq, 6), (lk, rk), (lk, rk)) for x in (h, d)]
    kw = dict(sm_scale=d**-0.5, kernel=2, causal=tpa.CAUSAL_BOTTOM_RIGHT if causal else False)
    o, lse = tpa.tpa_factors(*args, kv_lengths=torch.tensor(lengths, dtype=torch.int32, device=gpu), **kw)
    for i, n in enumerate(lengths):
        want, want_lse = tpa.tpa_factors(
            *(x[i : i + 1] for x in args), kv_lengths=torch.tensor([n], dtype=torch.int32, device=gpu), use_workspace=False, **kw)
        assert torch.equal(lse[i].isinf(), want_lse[0].isinf())
        assert torch.equal(o[i].isnan(), want[0].isnan())
        got, want = o[i].float().nan_to_num(), want[0].float().nan_to_num()
        # K and V are rounded to bf16 on either route, sums and results once more: 2^-9 of each
        assert (got - want).norm() <= 6e-3 * want.norm()
        seen = ~want_lse[0].isinf()
        assert torch.allclose(lse[i][seen], want_lse[0][seen], atol=4e-3, rtol=0)
