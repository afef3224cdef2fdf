"""The merge of the key ranges where it changes form: as many ranges as one trip of 1, 2, 4 and 8 groups of threads takes, one
more, and several trips; heads that do not fill a block of threads; ranges without keys; rows without any."""

import pytest
import torch

from conftest import make_factors
from test_gpu_parity import BF16_TOL, F32_TOL, _varlen_reference, as_f64, bf16_bounds, check, to_gpu, tpa_split

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("h,d", [(8, 128), (24, 64), (40, 128)])
@pytest.mark.parametrize("splits", [1, 4, 5, 8, 9, 16, 17, 32, 33, 70])
def test_ranges_merged(gpu, dt, h, d, splits):
    from tpa import tpa

    lengths, lk = [1500, 70, 1], 1500  # the shorter entries leave most ranges without keys
    q, k, v = (to_gpu(x, dt, gpu) for x in make_factors(71, len(lengths), 2, lk, h, d, d, 6, 2, scale_by_rank=True))
    kvl = torch.tensor(lengths, dtype=torch.int32)
    o, lse = tpa.tpa_decode(*tpa_split(q, k, v, h), sm_scale=d**-0.5, kv_lengths=kvl, num_splits=splits, kernel=2)
    o_ref, l_ref = _varlen_reference(as_f64(q), as_f64(k), as_f64(v), lengths, h, d**-0.5, False)
    bounds = bf16_bounds(q, k, v, h, d**-0.5, form="factored") if dt == torch.bfloat16 else None
    check(o, lse, o_ref, l_ref, BF16_TOL if dt == torch.bfloat16 else F32_TOL, bounds)


@pytest.mark.parametrize("b,lk", [(1, 4000), (2, 3000), (5, 2000), (40, 700)])
def test_rows_without_keys(gpu, b, lk):
    """Ranges dealt by length: an entry without keys has nan and -inf, as one that is alone, and its neighbours do not notice."""
    from tpa import tpa

    h, d = 16, 128
    q, k, v = (to_gpu(x, torch.bfloat16, gpu) for x in make_factors(72, b + 1, 1, lk, h, d, d, 6, 2, scale_by_rank=True))
    lengths = [lk - 3 * i for i in range(b)] + [0]
    args = dict(sm_scale=d**-0.5, kernel=2)
    o, lse = tpa.tpa_decode(*tpa_split(q, k, v, h), kv_lengths=torch.tensor(lengths, dtype=torch.int32), **args)
    assert torch.isneginf(lse[b]).all() and not torch.isfinite(o[b]).any()
    for i in range(0, b, 7):
        oi, li = tpa.tpa_decode(*tpa_split(q[i : i + 1], k[i : i + 1, : lengths[i]], v[i : i + 1, : lengths[i]], h), num_splits=1, **args)
        torch.testing.assert_close(o[i : i + 1], oi, rtol=2.0**-7, atol=1e-3)
        torch.testing.assert_close(lse[i : i + 1], li, rtol=0, atol=1e-4)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("splits", [0, 6, 9, 24])
def test_infinity_of_the_last_range(gpu, dt, splits):
    """A trip repeats the last range where there are no more: an infinity in it counts once and stays one."""
    from tpa import tpa

    h, d, lk = 16, 128, 1500
    q, k, v = (to_gpu(x, dt, gpu) for x in make_factors(73, 1, 1, lk, h, d, d, 6, 2, scale_by_rank=True))
    args = tpa_split(q, k, v, h)
    base, _ = tpa.tpa_decode(*args, sm_scale=d**-0.5, num_splits=splits, kernel=2)
    v[0, -1, 0, h] = float("inf")  # token factor of rank 0, its first element
    o, lse = tpa.tpa_decode(*tpa_split(q, k, v, h), sm_scale=d**-0.5, num_splits=splits, kernel=2)
    sign = torch.sign(v[0, -1, 0, :h].float())
    assert torch.equal(o[0, 0, :, 0].float(), sign * float("inf"))
    assert torch.equal(o[..., 1:], base[..., 1:])
