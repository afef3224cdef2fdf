"""The matrix-core backward at head size 64 works in blocks of 128 rows (documents, a causal mask of at most 2816 rows, few
workgroups, or fewer rounds of them) or 256 (everything else): sizes on either side of the blocks, of the 64-row tiles
and of those lines, with documents that share tiles and, in one case, ids that come back; against the oracle."""

import numpy as np
import pytest
import torch

from conftest import make_factors
from oracle import tpa_oracle as orc

pytestmark = pytest.mark.gpu


def _ids(kind, b, t):
    pos = np.arange(t)[None] + 17 * np.arange(b)[:, None]
    if kind == "documents":
        return (pos // 45).astype(np.int32)
    return (pos // 30 % 3).astype(np.int32)  # every id comes back: a wave's own range tells little


@pytest.mark.parametrize(
    "b,t,h,causal,kind",
    [
        (1, 65, 8, True, None),
        (2, 127, 8, True, "documents"),
        (1, 129, 8, False, "documents"),
        (1, 300, 8, True, "again"),
        (1, 257, 16, False, "again"),
        (3, 385, 8, True, None),
        (1, 2304, 8, True, None),
        (1, 2305, 8, True, None),
        (3, 2817, 8, True, None),    # blocks of 256: 576 workgroups of them
        (1, 600, 8, False, None),    # one round of blocks of 256
        (4, 512, 32, False, None),   # blocks of 256: two rounds, as four of half the size
        (5, 512, 32, False, None),   # three rounds against five
    ],
)
def test_backward_at_the_edges_of_blocks(gpu, b, t, h, causal, kind):
    from tpa import tpa

    d, scale = 64, 64**-0.5
    q, k, v = make_factors(31, b, t, t, h, d, d, 6, 2, scale_by_rank=True)
    do = np.random.default_rng(32).standard_normal((b, t, h, d)).astype(np.float32)
    ids = None if kind is None else _ids(kind, b, t)
    tq, tk, tv = (torch.from_numpy(x).to(gpu).to(torch.bfloat16).requires_grad_() for x in (q, k, v))
    tdo = torch.from_numpy(do).to(gpu).to(torch.bfloat16)
    tid = None if ids is None else torch.from_numpy(ids).to(gpu)
    tpa.tpa(tq, tk, tv, h, tid, tid, sm_scale=scale, causal=causal).backward(tdo)
    f64 = lambda x: x.detach().float().cpu().numpy().astype(np.float64)
    want = orc.tpa_backward(f64(tq), f64(tk), f64(tv), ids, ids, h, f64(tdo), sm_scale=scale, causal=causal)
    for name, x, w in zip("qkv", (tq, tk, tv), want):
        got = f64(x.grad)
        assert np.isfinite(got).all(), name
        # bf16 results (2^-9 relative) of bf16 probabilities and dS, and the bf16 o in delta
        assert np.abs(got - w).max() <= 2e-2 * np.abs(w).max(), name
