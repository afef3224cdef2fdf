"""Decode of eight heads, whose workgroups serve four query rows each: the ranges that are chosen for that fit the workspace that
callers are told, whichever form of the kernel reads the cache, and give the generic kernel's result."""

import pytest
import torch

from conftest import make_factors
from test_gpu_parity import to_gpu, tpa_split

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lengths", [False, True])
@pytest.mark.parametrize("descending", [False, True])
@pytest.mark.parametrize("b,lq,lk", [(1, 3, 5000), (1, 4, 16411), (3, 5, 1023), (2, 9, 4096), (64, 4, 300)])
def test_ranges_fit_the_workspace_told(gpu, b, lq, lk, descending, lengths):
    from tpa import _dispatch as dd
    from tpa import tpa

    h, d, rq, rk = 8, 64, 6, 2
    q, k, v = make_factors(61, b, lq, lk, h, d, d, rq, rk, scale_by_rank=True)
    qa, qb, *kv = (x.contiguous() for x in tpa_split(*(to_gpu(x, torch.bfloat16, gpu) for x in (q, k, v)), h))
    ends = torch.tensor([max(lq, lk - 401 * i) for i in range(b)], dtype=torch.int32, device=gpu)
    lib = dd.load_library()
    told, guard = tpa.decode_workspace_bytes(b, lq, lk, h, d), 1 << 16
    ws = torch.full((told + guard,), 0x7F, dtype=torch.uint8, device=gpu)

    def call(kernel, factors):
        o = torch.empty((b, lq, h, d), dtype=torch.bfloat16, device=gpu)
        lse = torch.empty((b, h, lq), dtype=torch.float32, device=gpu)
        args = dd.TpaFwdArgs(
            qa=dd.factor(qa), qb=dd.factor(qb), ka=factors[0], kb=factors[1], va=factors[2], vb=factors[3], o=o.data_ptr(), lse=lse.data_ptr(),
            B=b, lq=lq, lk=lk, H=h, dk=d, dv=d, rq=rq, rk=rk, dtype=dd.dtype_code(torch.bfloat16), sm_scale=d**-0.5, kernel=kernel,
            causal=tpa.CAUSAL_BOTTOM_RIGHT, workspace=ws.data_ptr(), workspace_bytes=told, kv_lengths=ends.data_ptr() if lengths else None)
        dd.check("tpa_decode", lib.tpa_decode(args, dd.current_stream_ptr(gpu)))
        torch.cuda.synchronize()
        return o, lse

    want = call(dd.KERNEL_GENERIC, [dd.factor(x) for x in kv])
    factors, flipped = [dd.factor(x) for x in kv], [x.flip(1, 2).contiguous() for x in kv]
    if descending:  # an address per lane, and two rows per workgroup
        factors = [dd.TpaFactor(f.data_ptr() + (lk * rk - 1) * x.shape[3] * 2, x.stride(0), -x.stride(1), -x.stride(2)) for f, x in zip(flipped, kv)]
    got = call(dd.KERNEL_MFMA, factors)
    assert (ws[told:] == 0x7F).all()
    for x, y in zip(got, want):
        # bf16 factors and results, probabilities rounded once: 2^-7 of results of order one, as the other decode tests have it
        torch.testing.assert_close(x.float(), y.float(), rtol=2e-2, atol=2e-2)
