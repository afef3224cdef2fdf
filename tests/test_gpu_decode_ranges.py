"""tpa_decode with key ranges dealt by the lengths of the batch entries, and with one count for all entries, against the
CPU oracle: one entry and as many as a wave has lanes (and one more, where all entries get one count again), lengths
from none to the whole cache, two row groups, ranks of the queries past one matrix instruction (16)."""

import pytest
import torch

from conftest import make_factors
from test_gpu_parity import BF16_TOL, F32_TOL, _varlen_reference, as_f64, bf16_bounds, check, to_gpu, tpa_split

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize(
    "lengths,lk,h,d,rq,rk",
    [
        ([3000], 4096, 16, 128, 6, 2),
        ([5], 4096, 8, 64, 17, 2),
        ([2000, 0, 17, 256], 2000, 40, 64, 16, 4),       # two head blocks; an entry without keys
        ([1 + 29 * i for i in range(64)], 1900, 8, 64, 6, 2),
        ([1] * 63 + [1500], 1500, 8, 64, 33, 8),          # one long entry among short ones
        ([700 + i for i in range(65)], 800, 8, 64, 1, 2),  # more entries than lanes
        (None, 1100, 8, 64, 6, 2),                        # 48 entries: five ranges each, not six
    ],
)
def test_ranges_dealt_by_length(gpu, dt, lengths, lk, h, d, rq, rk):
    from tpa import tpa

    b = 48 if lengths is None else len(lengths)
    q, k, v = make_factors(91, b, 1, lk, h, d, d, rq, rk, scale_by_rank=True)
    tq, tk, tv = (to_gpu(x, dt, gpu) for x in (q, k, v))
    for bi, n in enumerate(lengths or []):
        tk[bi, n:] = float("nan")
        tv[bi, n:] = float("nan")
    kvl = None if lengths is None else torch.tensor(lengths, dtype=torch.int32)
    o, lse = tpa.tpa_decode(*tpa_split(tq, tk, tv, h), sm_scale=d**-0.5, kv_lengths=kvl, kernel=2)
    o_ref, l_ref = _varlen_reference(as_f64(tq), as_f64(tk), as_f64(tv), lengths or [lk] * b, h, d**-0.5, False)
    tk, tv = tk.nan_to_num(), tv.nan_to_num()
    check(o, lse, o_ref, l_ref, BF16_TOL if dt == torch.bfloat16 else F32_TOL,
          bf16_bounds(tq, tk, tv, h, d**-0.5, form="factored") if dt == torch.bfloat16 else None)


@pytest.mark.parametrize("lq", [2, 3, 9])
def test_several_rows_are_the_rows_alone(gpu, lq):
    """Rows aligned with the end of each entry's keys: row i of `lq` sees what one row sees whose entry ends there."""
    from tpa import tpa

    lengths, lk, h, d = [40, 1000, 2047, 1500, 333], 2048, 8, 128
    b = len(lengths)
    q, k, v = make_factors(93, b, lq, lk, h, d, d, 6, 2, scale_by_rank=True)
    tq, tk, tv = (to_gpu(x, torch.bfloat16, gpu) for x in (q, k, v))
    kvl = torch.tensor(lengths, dtype=torch.int32)
    o, lse = tpa.tpa_decode(*tpa_split(tq, tk, tv, h), sm_scale=d**-0.5, kv_lengths=kvl, causal=tpa.CAUSAL_BOTTOM_RIGHT, kernel=2)
    bounds = bf16_bounds(tq, tk, tv, h, d**-0.5, form="factored")
    for i in range(lq):
        ends = [n - lq + 1 + i for n in lengths]
        o_ref, l_ref = _varlen_reference(as_f64(tq[:, i : i + 1]), as_f64(tk), as_f64(tv), ends, h, d**-0.5, False)
        check(o[:, i : i + 1], lse[:, :, i : i + 1], o_ref, l_ref, BF16_TOL, tuple(x[:, i : i + 1] for x in bounds))
