"""fp32 matrix-core kernels of 128 and 256 rows, forward and backward, over packed documents: a wave leaves out the tiles that
hold none of its own documents, also where ids come back or fall; against the oracle, with the bounds of the other fp32 tests."""

import numpy as np
import pytest
import torch

from conftest import make_factors
from oracle import tpa_oracle as orc
from test_gpu_backward import rel_err
from test_gpu_backward_blocks import _ids

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(
    "b,t,h,d,causal,kind",
    [
        (6, 257, 24, 64, False, "documents"),  # 256 rows forward, eight waves backward
        (6, 257, 24, 64, False, "again"),
        (4, 200, 40, 64, True, "falling"),     # 256 rows forward, four waves backward
        (2, 500, 32, 64, False, "documents"),  # 128 rows forward
        (5, 100, 64, 128, False, "again"),     # tiles of 32
        (6, 193, 32, 128, True, "documents"),
    ],
)
def test_documents(gpu, b, t, h, d, causal, kind):
    from tpa import tpa

    ids = -_ids("documents", b, t) if kind == "falling" else _ids(kind, b, t)
    q, k, v = make_factors(81, b, t, t, h, d, d, 6, 2, scale_by_rank=True)
    do = np.random.default_rng(82).standard_normal((b, t, h, d)).astype(np.float32)
    tq, tk, tv, tdo = (torch.from_numpy(x).to(gpu) for x in (q, k, v, do))
    tid, scale = torch.from_numpy(ids).to(gpu), d**-0.5
    sp = lambda x: (x[..., :h].contiguous(), x[..., h:].contiguous())
    o, lse = tpa.tpa_factors(*sp(tq), *sp(tk), *sp(tv), tid, tid, scale, causal, kernel=2)
    o_ref, l_ref = orc.tpa_reference(q.astype(np.float64), k.astype(np.float64), v.astype(np.float64), ids, ids, h, sm_scale=scale, causal=causal)
    assert np.abs(o.cpu().numpy() - o_ref).max() <= 1e-4
    assert np.abs(lse.cpu().numpy().transpose(0, 2, 1) - l_ref).max() <= 1e-3
    grads = tpa.tpa_factors_bwd(*sp(tq), *sp(tk), *sp(tv), tid, tid, o, lse, tdo, scale, causal, kernel=2)
    want = orc.tpa_backward(q, k, v, ids, ids, h, do, sm_scale=scale, causal=causal)
    for n, w in enumerate(want):
        got = np.concatenate([g.cpu().numpy() for g in grads[2 * n : 2 * n + 2]], axis=-1)
        assert rel_err(got, w) <= 2e-4, "qkv"[n]
