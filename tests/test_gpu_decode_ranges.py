"""tpa_decode with key ranges dealt by the lengths of the batch entries, and with one count for all entries, against the
CPU oracle: one entry and as many as a wave has lanes (and one more, where all entries get one count again), lengths
from none to the whole cache, two row groups, ranks of the queries past one matrix instruction (16)."""

import numpy as np
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


def _planned_ranges(lengths, lk, slots, min_keys):
    """Ranges per entry as the kernels plan them, in the same fp32 steps."""
    f = np.float32
    n = np.minimum(np.maximum(np.asarray(lengths), 0), lk)
    total = f(n.sum())
    shortest = max(total / f(slots), f(min_keys))
    longest = max(total / f(slots - len(n)) + f(1), shortest) if slots > len(n) else f(lk)
    for lane in range(64):  # the product and the sum round once, together: long double holds the product exactly
        length = f(np.longdouble((longest - shortest) * f(lane)) * np.longdouble(f(1) / f(63)) + np.longdouble(shortest))
        ranges = np.maximum(1, np.ceil(n.astype(f) * (f(1) / length))).astype(int)
        if ranges.sum() <= slots:
            return ranges
    return np.ones(len(n), int)


@pytest.mark.parametrize("seed", range(12))
def test_both_kernels_follow_the_stated_plan(gpu, seed):
    """The decode kernel and the merge work the plan out separately.  A workspace of NaN shows the first one's ranges (those
    that were written); a merge that takes others reads NaN."""
    from tpa import tpa

    rng = np.random.default_rng(seed)
    b, lk, h, d = int(rng.integers(1, 65)), int(rng.integers(300, 9000)), 8, 64
    lengths = rng.integers(0 if seed % 2 else lk // 2, lk + 1, b)
    lengths[0] = max(1, lengths[0])
    q, k, v = make_factors(97 + seed, b, 1, lk, h, d, d, 2, 2, scale_by_rank=True)
    parts = tpa_split(*(to_gpu(x, torch.bfloat16, gpu) for x in (q, k, v)), h)
    kvl = torch.tensor(lengths, dtype=torch.int32, device=gpu)
    default = tpa._d.load_library().tpa_decode_default_splits(b, 1, lk, h)
    slots = min(max(b, 256), b * default)
    ws = torch.full((tpa.decode_workspace_bytes(b, 1, lk, h, d),), 0xFF, dtype=torch.uint8, device=gpu)
    got = tpa.tpa_decode(*parts, sm_scale=d**-0.5, kv_lengths=kvl, kernel=2, workspace=ws)
    maxima = ws.view(torch.float32)[slots * h * d :][: slots * h].view(slots, h)
    written = (~maxima.isnan()).all(1).sum().item()
    assert written == _planned_ranges(lengths, lk, slots, 64).sum(), (b, lk, slots)
    want = tpa.tpa_decode(*parts, sm_scale=d**-0.5, kv_lengths=kvl, kernel=1)
    some = torch.from_numpy(lengths > 0).to(gpu)
    for x, y in zip(got, want):
        assert x[some].isfinite().all()
        torch.testing.assert_close(x[some].float(), y[some].float(), rtol=2e-2, atol=2e-2)
