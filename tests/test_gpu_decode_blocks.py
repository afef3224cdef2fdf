"""The split-key decode kernels where their loop and the query's ranks change form: no, one, two, three and four blocks per wave
with rows left over, ranks of the queries around half an operand (8) and a whole one (16), pages of a size that is and is not
a power of two, against the CPU oracle."""

import pytest
import torch

from conftest import make_factors
from test_gpu_parity import BF16_TOL, _varlen_reference, as_f64, bf16_bounds, check, to_gpu, tpa_split

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h,d,rk", [(16, 128, 2), (40, 64, 4), (40, 64, 8), (40, 64, 16)])
@pytest.mark.parametrize("rq", [1, 8, 9, 16, 17, 33])
@pytest.mark.parametrize("lq", [1, 2, 3])
@pytest.mark.parametrize("page", [0, 48, 64])
def test_blocks_per_wave(gpu, h, d, rk, rq, lq, page):
    from tpa import tpa

    per_wave = 4 * 32 // rk  # keys of one block per wave of a range
    lengths = [0, 1, per_wave // 4, per_wave - 1, per_wave + 1, 2 * per_wave, 3 * per_wave - 5, 4 * per_wave]
    b, lk = len(lengths), 4 * per_wave
    q, k, v = make_factors(97, b, lq, lk, h, d, d, rq, rk, scale_by_rank=True)
    tq, tk, tv = (to_gpu(x, torch.bfloat16, gpu) for x in (q, k, v))
    o_ref, l_ref = _varlen_reference(as_f64(tq), as_f64(tk), as_f64(tv), lengths, h, d**-0.5, False)
    bounds = bf16_bounds(tq, tk, tv, h, d**-0.5, form="factored")
    qa, qb, *kv = tpa_split(tq, tk, tv, h)
    table = None
    for bi, n in enumerate(lengths):  # nothing past the end of an entry is used
        for x in kv:
            x[bi, n:] = float("nan")
    if page:
        per_seq = -(-lk // page)
        order = torch.randperm(b * per_seq, generator=torch.Generator().manual_seed(5))
        table = order.to(torch.int32).view(b, per_seq)
        pools = []
        for x in kv:
            pool = torch.full((b * per_seq, page, *x.shape[2:]), float("nan"), dtype=x.dtype, device=x.device)
            for bi in range(b):
                for pi in range(per_seq):
                    part = x[bi, pi * page : (pi + 1) * page]
                    pool[int(table[bi, pi]), : part.shape[0]] = part
            pools.append(pool)
        kv, table = pools, table.to(gpu)
        for bi, n in enumerate(lengths):  # entries of the table past an entry's last page are not followed
            table[bi, max(0, -(-n // page)) :] = -(1 << 30)
    kvl = torch.tensor(lengths, dtype=torch.int32)
    o, lse = tpa.tpa_decode(qa, qb, *kv, sm_scale=d**-0.5, num_splits=1, kv_lengths=kvl, page_table=table, kernel=2)
    check(o, lse, o_ref, l_ref, BF16_TOL, bounds)


@pytest.mark.parametrize("lq", [1, 2, 3])
@pytest.mark.parametrize("page", [0, 16])
@pytest.mark.parametrize("order", ["far apart", "descending"])
def test_rows_that_lie_far_apart_or_descend(gpu, order, page, lq):
    """Rows of the cache more than 2^25 elements apart, or in descending order, give what the same rows next to each other give."""
    from tpa import _dispatch as dd

    b, lk, h, d, rq, rk, far = 2, 80, 16, 64, 6, 2, (1 << 25) + 8
    q, k, v = (to_gpu(x, torch.bfloat16, gpu) for x in make_factors(98, b, lq, lk, h, d, d, rq, rk, scale_by_rank=True))
    qa, qb, *kv = (x.contiguous() for x in tpa_split(q, k, v, h))
    lengths = torch.tensor([lk, 37], dtype=torch.int32, device=gpu)
    table = None
    if page:
        kv = [x.view(b * lk // page, page, rk, x.shape[-1]) for x in kv]
        table = torch.arange(b * lk // page, dtype=torch.int32, device=gpu).view(b, -1)
    lib = dd.load_library()
    ws = torch.empty(1 << 24, dtype=torch.uint8, device=gpu)

    def call(factors):
        o = torch.empty((b, lq, h, d), dtype=torch.bfloat16, device=gpu)
        lse = torch.empty((b, h, lq), dtype=torch.float32, device=gpu)
        args = dd.TpaFwdArgs(
            qa=dd.factor(qa), qb=dd.factor(qb), ka=factors[0], kb=factors[1], va=factors[2], vb=factors[3], o=o.data_ptr(), lse=lse.data_ptr(),
            B=b, lq=lq, lk=lk, H=h, dk=d, dv=d, rq=rq, rk=rk, dtype=dd.dtype_code(torch.bfloat16), sm_scale=d**-0.5, kernel=dd.KERNEL_MFMA,
            workspace=ws.data_ptr(), workspace_bytes=ws.numel(), num_splits=1, kv_lengths=lengths.data_ptr(),
            page_table=table.data_ptr() if page else None, page_size=page, pages_per_seq=lk // page if page else 0)
        dd.check("tpa_decode", lib.tpa_decode(args, dd.current_stream_ptr(gpu)))
        torch.cuda.synchronize()
        return o, lse

    want = call([dd.factor(x) for x in kv])
    moved = []
    for n, x in enumerate(kv):
        if order == "descending":
            flipped = x.flip(1, 2).contiguous()
            last = (x.shape[1] * rk - 1) * x.shape[3] * 2
            moved.append((flipped, dd.TpaFactor(flipped.data_ptr() + last, x.stride(0), -x.stride(1), -x.stride(2))))
        elif n == 1:  # one array is enough for the far form; batch entries (pages) lie between its rows
            place = torch.empty((x.shape[1] * rk - 1) * far + x.shape[0] * d, dtype=x.dtype, device=gpu)
            spread = place.as_strided(x.shape, (d, rk * far, far, 1))
            spread.copy_(x)
            moved.append((spread, dd.factor(spread)))
        else:
            moved.append((x, dd.factor(x)))
    got = call([f for _, f in moved])
    for x, y in zip(got, want):
        torch.testing.assert_close(x, y, rtol=2.0**-7, atol=1e-3)
