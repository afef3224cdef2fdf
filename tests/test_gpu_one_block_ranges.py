"""bf16 forward of one block of query rows over fewer than 1536 keys, the keys split over workgroups: which calls ask for the room of the
partial results (no GPU needed), and that the results agree with those of the call that has none, at ranges that end up empty too."""

import ctypes

import numpy as np
import pytest
import torch

from test_abi import _forward_call


@pytest.mark.parametrize(
    "B,H,D,lq,lk,rk,ranges",
    [
        (1, 8, 128, 140, 1160, 2, 7),
        (2, 32, 128, 140, 1160, 2, 4),
        (2, 32, 128, 100, 700, 2, 1),
        (8, 16, 128, 256, 1160, 2, 1),
        (16, 16, 128, 17, 1160, 2, 1),
        (1, 8, 64, 140, 1160, 2, 7),
        (1, 8, 64, 100, 520, 2, 1),
        (1, 8, 128, 257, 1160, 2, 1),  # two blocks
        (1, 8, 128, 140, 1160, 4, 7),
        (1, 8, 64, 100, 700, 4, 1),
    ],
)
def test_which_calls_ask_for_it(B, H, D, lq, lk, rk, ranges):
    from tpa import _dispatch as d

    lib = d.load_library()
    fake = d.TpaFactor(256, 8, 8, 8)
    need = []
    for splits in (0, 1):
        call = _forward_call(B=B, H=H, D=D, lq=lq, lk=lk, rk=rk, qa=fake, qb=fake, ka=fake, kb=fake, va=fake, vb=fake, num_splits=splits)
        need.append(lib.tpa_fwd_call_workspace_bytes(ctypes.byref(call)))
    assert need[0] - need[1] == (ranges * B * lq * H * (D + 2) * 4 if ranges > 1 else 0)
    assert need[0] <= lib.tpa_fwd_best_workspace_bytes(B, lq, lk, H, D, D, 6, rk)


@pytest.mark.parametrize(
    "lq,lk,rk,mask,ranges",
    [
        (100, 1400, 2, dict(causal=1), 1),                        # two tiles are in reach
        (100, 1400, 4, dict(causal=1), 1),
        (100, 1400, 2, dict(causal=1, causal_offset=1300), 8),
        (100, 1400, 2, dict(causal=1, causal_offset=700), 7),     # 13 tiles, two for each
        (100, 1400, 2, dict(causal=1, causal_offset=-50), 1),
        (100, 1400, 2, dict(causal=2), 8),
        (100, 1400, 2, dict(), 8),
        (64, 448, 2, dict(), 1),                                  # dense tiles, of which seven are not worth it
    ],
)
def test_keys_behind_the_mask_ask_for_no_ranges(lq, lk, rk, mask, ranges):
    from tpa import _dispatch as d

    lib = d.load_library()
    fake = d.TpaFactor(256, 8, 8, 8)
    need = []
    for splits in (0, 1):
        call = _forward_call(B=1, H=8, D=128, lq=lq, lk=lk, rk=rk, qa=fake, qb=fake, ka=fake, kb=fake, va=fake, vb=fake, num_splits=splits, **mask)
        need.append(lib.tpa_fwd_call_workspace_bytes(ctypes.byref(call)))
    assert need[0] - need[1] == (ranges * lq * 8 * (128 + 2) * 4 if ranges > 1 else 0)
    assert need[0] <= lib.tpa_fwd_best_workspace_bytes(1, lq, lk, 8, 128, 128, 6, rk)


@pytest.mark.gpu
@pytest.mark.parametrize("mask", ["none", "top left", "bottom right", "lengths"])
@pytest.mark.parametrize("b,h,d,lq,lk,rk", [(5, 1, 128, 140, 1160, 2), (5, 1, 64, 256, 900, 2), (2, 8, 128, 17, 520, 2), (1, 8, 128, 100, 1400, 4)])
def test_results_agree(gpu, b, h, d, lq, lk, rk, mask):
    """Rank 2: the same arithmetic, merged with exact powers of two, so that only fp32 sums and the last rounding to 8 bits differ (2^-8
    of a value).  Rank 4 takes the dense arrays beside it: either route rounds to 8 bits at four places, as that route's own test has it."""
    from tpa import tpa

    gen = torch.Generator(device="cpu").manual_seed(lk)
    make = lambda l, r, x: (torch.randn((b, l, r, x), generator=gen) / r**0.5).to(gpu, torch.bfloat16)
    args = [make(l, r, x) for l, r in ((lq, 6), (lk, rk), (lk, rk)) for x in (h, d)]
    kw = dict(sm_scale=d**-0.5, causal=mask == "top left", kernel=2)
    if mask in ("lengths", "bottom right"):
        kw["kv_lengths"] = torch.tensor([lk, 0, 1, 64, lk - 100][:b], dtype=torch.int32, device=gpu)
    if mask == "bottom right":
        kw["causal"] = tpa.CAUSAL_BOTTOM_RIGHT
    (o1, l1), (o2, l2) = (tpa.tpa_factors(*args, use_workspace=w, **kw) for w in (True, False))
    x, y = (o.float().cpu().numpy().astype(np.float64) for o in (o1, o2))
    np.testing.assert_array_equal(np.isnan(x), np.isnan(y))
    assert np.nanmax(np.abs(x - y)) <= (2**-8 if rk == 2 else 2**-6) * np.nanmax(np.abs(y))
    a, c = (l.cpu().numpy() for l in (l1, l2))
    seen = np.isfinite(c)
    np.testing.assert_array_equal(np.isfinite(a), seen)
    assert np.abs(a[seen] - c[seen]).max() <= (1e-5 if rk == 2 else 2**-6)
