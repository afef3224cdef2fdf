"""Decode of 8 and 16 heads, where 32 / H query rows share the columns of a matrix instruction: a full set, one that is not
full, and several of them, with keys that end inside blocks, pages and the causal limit of the last rows.  Columns share no
arithmetic, so every row is bit for bit what the call gives for that row alone, also beside a row that is not finite."""

import pytest
import torch

from conftest import make_factors
from test_gpu_parity import to_gpu, tpa_split

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h,d,rk", [(8, 64, 1), (8, 128, 2), (8, 64, 8), (16, 64, 4), (16, 128, 2), (16, 128, 32)])
@pytest.mark.parametrize("rq", [6, 17])
@pytest.mark.parametrize("lq", [2, 3, 4, 5, 9])
def test_rows_side_by_side_are_the_rows_alone(gpu, h, d, rk, rq, lq):
    from tpa import tpa

    b, lk, page, splits = 3, 384, 64, 2
    q, k, v = (to_gpu(x, torch.bfloat16, gpu) for x in make_factors(55, b, lq, lk, h, d, d, rq, rk, scale_by_rank=True))
    bad = lq // 2
    q[0, bad] = float("inf")
    q[1, bad] = float("nan")
    qa, qb, *kv = tpa_split(q, k, v, h)
    kv = [x.contiguous() for x in kv]
    lengths = [lk, 201, lq]
    table = torch.arange(b * lk // page, dtype=torch.int32, device=gpu).view(b, -1)
    pools = [x.view(b * lk // page, page, rk, x.shape[-1]) for x in kv]

    def call(rows, ends, causal, paged):
        return tpa.tpa_decode(
            qa[:, rows], qb[:, rows], *(pools if paged else kv), sm_scale=d**-0.5, num_splits=splits, causal=causal, kernel=2,
            kv_lengths=torch.tensor(ends, dtype=torch.int32, device=gpu), page_table=table if paged else None)

    for paged in (False, True):
        o, lse = call(slice(0, lq), lengths, tpa.CAUSAL_BOTTOM_RIGHT, paged)
        for i in range(lq):
            oi, li = call(slice(i, i + 1), [n - lq + 1 + i for n in lengths], False, paged)
            torch.testing.assert_close(o[:, i : i + 1], oi, rtol=0, atol=0, equal_nan=True)
            torch.testing.assert_close(lse[:, :, i : i + 1], li, rtol=0, atol=0, equal_nan=True)
            assert i == bad or torch.isfinite(oi).all()
