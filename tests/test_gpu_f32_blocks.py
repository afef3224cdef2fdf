"""fp32 matrix-core kernels at the edges of the rule that picks the rows of a workgroup: 32 (its waves split the keys or
query rows), 128 or 256 forward, 32 or 128 backward - against the CPU oracle, forward and backward of one problem each.

Tolerances: fp32 arithmetic throughout, so the bounds are those of the other fp32 tests: 1e-4 on outputs and 1e-3 on the
logsumexp for factors of this size, 2e-4 of the largest entry on gradients.
"""

import numpy as np
import pytest
import torch

from conftest import make_factors, segment_ids
from oracle import tpa_oracle as orc
from test_gpu_backward import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(
    "b,lq,lk,h,d,rq,rk,causal,seg",
    [
        (1, 64, 64, 1, 64, 1, 1, False, None),     # two tiles of 32: two of the four waves have nothing
        (1, 97, 65, 3, 128, 4, 3, True, None),     # a tile of one key, an odd rank, fewer keys than rows
        (2, 65, 200, 2, 64, 6, 2, False, None),    # a block of one row
        (1, 160, 160, 2, 128, 2, 5, True, 33),     # windows that start inside a tile
        (1, 300, 300, 2, 64, 6, 2, False, 70),     # rows of two documents in a block
        (2, 1025, 1025, 8, 64, 2, 2, True, None),  # 528 blocks of 32 rows: 128-row workgroups forward, 32 backward
        (6, 257, 257, 24, 64, 2, 2, True, 100),    # 288 blocks of 256 rows: the largest workgroups, with windows
        (3, 300, 200, 32, 128, 1, 2, False, None), # 288 blocks of 128 rows backward
    ],
)
def test_f32_workgroup_sizes(gpu, b, lq, lk, h, d, rq, rk, causal, seg):
    from tpa import tpa

    q, k, v = make_factors(71, b, lq, lk, h, d, d, rq, rk, scale_by_rank=True)
    do = np.random.default_rng(72).standard_normal((b, lq, h, d)).astype(np.float32)
    qseg = segment_ids(lq, seg, b) if seg else None
    kvseg = segment_ids(lk, seg, b) if seg else None
    scale = d**-0.5
    tq, tk, tv, tdo = (torch.from_numpy(x).to(gpu) for x in (q, k, v, do))
    ids = [None if x is None else torch.from_numpy(x).to(gpu) for x in (qseg, kvseg)]
    sp = lambda t: (t[..., :h].contiguous(), t[..., h:].contiguous())
    o, lse = tpa.tpa_factors(*sp(tq), *sp(tk), *sp(tv), *ids, scale, causal, kernel=2)
    o_ref, l_ref = orc.tpa_reference(q.astype(np.float64), k.astype(np.float64), v.astype(np.float64), qseg, kvseg, h, sm_scale=scale, causal=causal)
    got_o, got_l = o.cpu().numpy().astype(np.float64), lse.cpu().numpy().astype(np.float64).transpose(0, 2, 1)
    np.testing.assert_array_equal(np.isnan(got_o), np.isnan(o_ref))
    np.testing.assert_array_equal(np.isneginf(got_l), np.isneginf(l_ref))
    assert np.nanmax(np.abs(got_o - o_ref)) <= 1e-4
    seen = ~np.isneginf(l_ref)
    assert np.max(np.abs(got_l[seen] - l_ref[seen])) <= 1e-3
    grads = tpa.tpa_factors_bwd(*sp(tq), *sp(tk), *sp(tv), *ids, o, lse, tdo, scale, causal, kernel=2)
    want = orc.tpa_backward(q, k, v, qseg, kvseg, h, do, sm_scale=scale, causal=causal)
    for n, w in enumerate(want):
        got = np.concatenate([g.cpu().numpy() for g in grads[2 * n : 2 * n + 2]], axis=-1)
        assert rel_err(got, w) <= 2e-4, "qkv"[n]
