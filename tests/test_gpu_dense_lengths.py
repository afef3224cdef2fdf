"""The dense arrays of a forward call hold no more keys than its lengths and its mask let a query see: whatever lies in the padding of the
cache and in the rest of the workspace, the results are the same bits."""

import pytest
import torch


@pytest.mark.gpu
@pytest.mark.parametrize("mask", ["lengths", "bottom right", "short offset", "before the keys", "packed"])
@pytest.mark.parametrize(
    "dtype,b,h,d,lq,lk,rk",
    [
        (torch.bfloat16, 5, 8, 64, 300, 700, 4),
        (torch.bfloat16, 5, 16, 128, 40, 1100, 8),
        (torch.bfloat16, 1, 8, 64, 33, 4000, 4),  # the keys in ranges
        (torch.bfloat16, 2, 8, 128, 600, 900, 2),
        (torch.float32, 5, 8, 64, 65, 705, 4),
        (torch.float32, 3, 16, 128, 140, 400, 3),
    ],
)
def test_nothing_beyond_is_met(gpu, dtype, b, h, d, lq, lk, rk, mask):
    from tpa import tpa

    gen = torch.Generator(device="cpu").manual_seed(lk)
    make = lambda l, r, x: (torch.randn((b, l, r, x), generator=gen) / r**0.5).to(gpu, dtype)
    args = [make(l, r, x) for l, r in ((lq, 6), (lk, rk), (lk, rk)) for x in (h, d)]
    kw = dict(sm_scale=d**-0.5, kernel=2, causal=mask in ("short offset", "before the keys"))
    ends = [lk] * b
    if mask == "short offset":
        kw["causal_offset"] = 77
        ends = [min(lk, lq + 77)] * b
    if mask == "before the keys":
        kw["causal_offset"] = -lq // 2
        ends = [min(lk, lq - -(-lq // 2))] * b
    if mask in ("lengths", "bottom right", "packed"):
        ends = [lk - 130, 1, 64, 65, 0][:b]
        kw["kv_lengths"] = torch.tensor(ends, dtype=torch.int32, device=gpu)
    if mask == "bottom right":
        kw["causal"] = tpa.CAUSAL_BOTTOM_RIGHT
    if mask == "packed":
        ids = (torch.arange(lk, dtype=torch.int32)[None] // 97).expand(b, lk).contiguous().to(gpu)
        kw["q_segment_ids"], kw["kv_segment_ids"] = ids[:, :lq].contiguous(), ids

    def run(filling):
        xs = list(args)
        for n in range(2, 6):
            xs[n] = xs[n].clone()
            for i, x in enumerate(ends):
                xs[n][i, x:] = filling
        # the allocator hands this block to the call
        torch.full((4 * 4 * b * h * d * (lq + 2 * lk),), filling, dtype=torch.float32, device=gpu)
        return tpa.tpa_factors(*xs, **kw)

    (o1, l1), (o2, l2) = run(0.0), run(float("nan"))
    assert torch.equal(l1, l2)
    assert torch.equal(o1.nan_to_num(nan=1e9), o2.nan_to_num(nan=1e9))
