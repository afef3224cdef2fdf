"""The rule that sends a forward call of rank 2 below 2048 rows through dense Q, K and V: which calls it takes (from the
workspace they ask for, no GPU needed), and that both routes give one result over the forms that it accepts.

Tolerance: both routes round Q, K, V, P and the result at the same places; fp32 sums of another order move a result by far
less than a bf16 spacing, so it may round to the neighbouring value: 2^-7 of its magnitude, or of the row's largest entries
times 2^-12 where terms cancel.  The logsumexp is fp32: 1e-5.
"""

import ctypes

import numpy as np
import pytest
import torch

from conftest import segment_ids
from test_abi import _forward_call


@pytest.mark.parametrize(
    "B,H,D,lq,lk,dense",
    [
        (1, 64, 128, 256, 256, False),   # one query block
        (1, 64, 128, 257, 257, False),   # 128 workgroups
        (1, 32, 128, 257, 257, True),    # 64
        (1, 32, 64, 257, 257, False),    # head size 64 not below 65
        (1, 32, 128, 257, 1285, True),
        (1, 32, 128, 257, 1286, False),  # more than five keys per row
        (13, 5, 128, 257, 257, False),   # 130
        (8, 16, 64, 999, 999, False),    # 512 workgroups, but short
        (8, 16, 64, 1000, 1000, True),
        (4, 16, 64, 1000, 1000, False),  # 256
        (1, 1, 64, 2048, 9000, True),    # by length, as ever
    ],
)
def test_which_calls_go_through_dense_arrays(B, H, D, lq, lk, dense):
    from tpa import _dispatch as d

    need = d.load_library().tpa_fwd_call_workspace_bytes(ctypes.byref(_forward_call(B=B, H=H, D=D, lq=lq, lk=lk, rk=2, num_splits=1)))
    slot = lambda n: (n * 2 + 255) // 256 * 256
    assert need == (slot(B * lq * H * D) + 2 * slot(B * lk * H * D) if dense else 0)


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["concatenated", "split", "ranks first"])
@pytest.mark.parametrize(
    "b,h,d,lq,lk,mask",
    [
        (1, 8, 128, 257, 257, "causal"),
        (2, 16, 128, 300, 301, "none"),
        (3, 8, 128, 391, 1777, "offset"),
        (5, 16, 64, 1000, 1000, "packed"),
        (9, 8, 64, 1001, 999, "causal"),
        (2, 40, 128, 1023, 1100, "lengths"),
    ],
)
def test_both_routes_agree(gpu, b, h, d, lq, lk, mask, layout):
    from tpa import tpa

    gen = torch.Generator(device="cpu").manual_seed(lq)

    def factors(l, r):
        x = (torch.randn((b, l, r, h + d), generator=gen) / r**0.5).to(gpu).to(torch.bfloat16)
        parts = x[..., :h], x[..., h:]
        if layout == "split":
            return tuple(p.contiguous() for p in parts)
        if layout == "ranks first":
            return tuple(p.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3) for p in parts)
        return parts

    args = factors(lq, 6) + factors(lk, 2) + factors(lk, 2)
    kw = dict(sm_scale=d**-0.5, causal=mask in ("causal", "offset", "packed"), kernel=2)
    if mask == "offset":
        kw["causal_offset"] = lk - lq
    if mask == "packed":
        kw["q_segment_ids"] = kw["kv_segment_ids"] = torch.from_numpy(segment_ids(lq, 231, b)).to(gpu)
    if mask == "lengths":
        kw["kv_lengths"] = torch.tensor([lk, lk - 77], dtype=torch.int32, device=gpu)
    (o1, l1), (o2, l2) = (tpa.tpa_factors(*args, use_workspace=w, **kw) for w in (True, False))
    x, y = (o.float().cpu().numpy().astype(np.float64) for o in (o1, o2))
    np.testing.assert_array_equal(np.isnan(x), np.isnan(y))
    slack = np.maximum(2.0**-7 * np.abs(y), 2.0**-12 * np.nanmax(np.abs(y), axis=-1, keepdims=True))
    assert not (np.abs(x - y) > slack).any()
    a, c = (l.cpu().numpy() for l in (l1, l2))
    seen = np.isfinite(c)
    np.testing.assert_array_equal(np.isfinite(a), seen)
    assert np.abs(a[seen] - c[seen]).max() <= 1e-5
