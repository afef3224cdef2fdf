"""One block of rows of rank 2 at head size 128 over dense arrays, on either side of the lines to the fused kernel: as without a workspace."""

import pytest
import torch


@pytest.mark.gpu
@pytest.mark.parametrize("option", ["none", "causal", "offset", "lengths", "documents"])
@pytest.mark.parametrize(
    "b,h,lq,lk,rq",
    [
        (1, 8, 17, 768, 6),
        (1, 8, 256, 1, 6),
        (1, 16, 255, 65, 16),
        (5, 8, 200, 400, 6),    # 40 000 elements of D, the most
        (5, 8, 202, 400, 6),    # fused
        (1, 8, 100, 769, 6),   # fused
        (2, 8, 60, 64, 5),      # fused: few ranks of Q
        (1, 12, 40, 200, 6),    # fused: no whole groups of heads
        (2, 16, 130, 500, 33),
    ],
)
def test_as_without_a_workspace(gpu, b, h, lq, lk, rq, option):
    from tpa import tpa

    d = 128
    gen = torch.Generator(device=gpu).manual_seed(lq + lk)
    make = lambda l, r, x: (torch.randn((b, l, r, x), generator=gen, device=gpu) / r**0.5).to(torch.bfloat16)
    args = [make(l, r, x) for l, r in ((lq, rq), (lk, 2), (lk, 2)) for x in (h, d)]
    kw = dict(sm_scale=d**-0.5)
    if option in ("causal", "offset"):
        kw.update(causal=True, causal_offset=max(0, lk - lq) if option == "offset" else 0)
    if option == "lengths":
        kw["kv_lengths"] = torch.tensor([lk * (i + 1) // b for i in range(b)], dtype=torch.int32, device=gpu)
    if option == "documents":
        ids = lambda l: (torch.arange(l, dtype=torch.int32, device=gpu)[None] // 70).expand(b, l).contiguous()
        kw.update(q_segment_ids=ids(lq), kv_segment_ids=ids(lk))
    o, lse = tpa.tpa_factors(*args, **kw)
    want, want_lse = tpa.tpa_factors(*args, use_workspace=False, **kw)
    assert torch.equal(lse.isinf(), want_lse.isinf())
    assert torch.equal(o.isnan(), want.isnan())
    o, want = o.float().nan_to_num(), want.float().nan_to_num()
    # Q, K and V are rounded to bf16 on either route, sums and results once more: 2^-9 of each
    assert (o - want).norm() <= 6e-3 * want.norm()
    seen = ~want_lse.isinf()
    assert torch.allclose(lse[seen], want_lse[seen], atol=4e-3, rtol=0)
