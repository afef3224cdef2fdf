"""tpa_fwd with the keys of a query block split over workgroups (few query rows over many keys), against the CPU oracle.

The partial results are merged with exact powers of two, so the split changes nothing but the order of fp32 sums: the
bounds are those of the unsplit bf16 kernels (tests/error_model.py).
"""

import ctypes

import numpy as np
import pytest
import torch

from conftest import make_factors
from oracle import tpa_oracle as orc
from test_gpu_parity import BF16_TOL, as_f64, bf16_bounds, check, to_gpu, visible_bias

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(
    "b,lq,lk,h,d,rq,rk,causal,splits",
    [
        (1, 100, 700, 2, 128, 6, 2, 0, 3),   # rank-2 loop, 11 tiles in ranges of 3 and 4
        (2, 300, 300, 3, 64, 6, 2, 1, 5),    # as many ranges as tiles: the first block's last ones are empty
        (1, 257, 1500, 2, 128, 3, 4, 2, 4),  # dense route, aligned with the end of the keys
        (1, 60, 1030, 8, 64, 4, 8, 0, 16),   # dense route for one block over many keys; a last tile of six keys
        (1, 40, 900, 1, 64, 2, 3, 1, 2),     # any-rank loader; every row sees keys of the first range only
        (1, 520, 520, 9, 128, 1, 2, 1, 2),   # an odd number of heads: no head groups
    ],
)
def test_split_prefill_matches_the_oracle(gpu, b, lq, lk, h, d, rq, rk, causal, splits):
    from tpa import _dispatch as disp

    lib = disp.load_library()
    q, k, v = make_factors(81, b, lq, lk, h, d, d, rq, rk, scale_by_rank=True)
    scale = d**-0.5
    tq, tk, tv = (to_gpu(x, torch.bfloat16, gpu) for x in (q, k, v))
    parts = [x.contiguous() for t in (tq, tk, tv) for x in (t[..., :h], t[..., h:])]
    o = torch.empty((b, lq, h, d), dtype=torch.bfloat16, device=gpu)
    lse = torch.empty((b, h, lq), dtype=torch.float32, device=gpu)
    dense = lib.tpa_fwd_workspace_bytes(b, lq, lk, h, d, d, rq, rk)
    ws = torch.empty(dense + splits * b * lq * h * (d + 2) * 4 + 256, dtype=torch.uint8, device=gpu)
    pad = (-ws.data_ptr()) % 256
    args = disp.TpaFwdArgs(
        **{n: disp.factor(x) for n, x in zip(("qa", "qb", "ka", "kb", "va", "vb"), parts)}, o=o.data_ptr(), lse=lse.data_ptr(),
        B=b, lq=lq, lk=lk, H=h, dk=d, dv=d, rq=rq, rk=rk, dtype=disp.TPA_DTYPE_BF16, sm_scale=scale, causal=causal, kernel=disp.KERNEL_MFMA,
        workspace=ws.data_ptr() + pad, workspace_bytes=ws.numel() - pad, num_splits=splits)
    assert lib.tpa_fwd(ctypes.byref(args), disp.current_stream_ptr(gpu)) == 0
    bias = np.zeros((b, lq, lk))
    if causal:
        bias[:] = np.where(np.tril(np.ones((lq, lk), bool), k=lk - lq if causal == 2 else 0), 0.0, -np.inf)
    o_ref, l_ref = orc.mha_forward(*[orc.reconstruct(*orc.split_factors(as_f64(t), h)) for t in (tq, tk, tv)], bias=bias, sm_scale=scale)
    check(o, lse, o_ref, l_ref, BF16_TOL, bf16_bounds(tq, tk, tv, h, scale))


def test_the_python_api_brings_the_workspace_for_it(gpu):
    """A chunk of 40 query rows over 3000 keys: the default choice splits the keys and agrees with the call that may not."""
    from tpa import tpa

    q, k, v = make_factors(83, 1, 40, 3000, 8, 128, 128, 6, 2, scale_by_rank=True)
    parts = [x for t in (q, k, v) for x in (to_gpu(t[..., :8], torch.bfloat16, gpu), to_gpu(t[..., 8:], torch.bfloat16, gpu))]
    a, la = tpa.tpa_factors(*parts, sm_scale=128**-0.5)
    c, lc = tpa.tpa_factors(*parts, sm_scale=128**-0.5, use_workspace=False)
    # fp32 sums in another order, rounded to bf16: at most one spacing apart
    assert torch.all((a.float() - c.float()).abs() <= 2.0**-7 * torch.maximum(a.float().abs(), c.float().abs()) + 1e-6)
    assert torch.allclose(la, lc, atol=1e-5)


@pytest.mark.parametrize("causal", [0, 1, 2])
@pytest.mark.parametrize(
    "lq,lk,h,d,rq,rk,lengths,splits",
    [
        (150, 900, 2, 128, 6, 2, (900, 0, 64, 65, 149, 151), 4),  # rank-2 loop; an entry without keys, ends of tiles, the diagonal
        (300, 700, 2, 64, 3, 2, (700, 300, 257, 1), 11),          # two blocks, as many ranges as tiles: most of a short entry's are empty
        (100, 1100, 8, 64, 4, 4, (1100, 0, 99, 640), 5),          # dense keys and values (one block over many keys)
        (270, 600, 3, 128, 2, 1, (33, 600, 271), 3),              # dense keys and values, odd number of heads
        (70, 500, 2, 64, 2, 3, (500, 0, 70), 2),                  # any-rank loader
    ],
)
def test_split_prefill_of_a_ragged_batch(gpu, lq, lk, h, d, rq, rk, lengths, splits, causal):
    """Chunks over caches of different lengths: padding of NaN is never read, a workspace of NaN shows no range that was not
    written, rows without a key (an empty entry; bottom-right aligned rows of entries shorter than the chunk) are NaN / -inf."""
    from tpa import _dispatch as disp

    lib, b = disp.load_library(), len(lengths)
    q, k, v = make_factors(85, b, lq, lk, h, d, d, rq, rk, scale_by_rank=True)
    scale = d**-0.5
    tq, tk, tv = (to_gpu(x, torch.bfloat16, gpu) for x in (q, k, v))
    padded = [t.clone() for t in (tk, tv)]
    for t in padded:
        for bi, n in enumerate(lengths):
            t[bi, n:] = float("nan")
    parts = [x.contiguous() for t in (tq, *padded) for x in (t[..., :h], t[..., h:])]
    kvl = torch.tensor(lengths, dtype=torch.int32, device=gpu)
    o = torch.empty((b, lq, h, d), dtype=torch.bfloat16, device=gpu)
    lse = torch.empty((b, h, lq), dtype=torch.float32, device=gpu)
    args = disp.TpaFwdArgs(
        **{n: disp.factor(x) for n, x in zip(("qa", "qb", "ka", "kb", "va", "vb"), parts)}, o=o.data_ptr(), lse=lse.data_ptr(),
        B=b, lq=lq, lk=lk, H=h, dk=d, dv=d, rq=rq, rk=rk, dtype=disp.TPA_DTYPE_BF16, sm_scale=scale, causal=causal, kernel=disp.KERNEL_MFMA,
        kv_lengths=kvl.data_ptr(), num_splits=splits)
    need = lib.tpa_fwd_call_workspace_bytes(ctypes.byref(args))
    assert need >= splits * b * lq * h * (d + 2) * 4
    ws = torch.full((need + 256,), 0xFF, dtype=torch.uint8, device=gpu)
    args.workspace, args.workspace_bytes = ws.data_ptr() + (-ws.data_ptr()) % 256, need
    assert lib.tpa_fwd(ctypes.byref(args), disp.current_stream_ptr(gpu)) == 0
    bias = visible_bias(b, lq, lk, causal=bool(causal), lengths=lengths, bottom_right=causal == 2)
    o_ref, l_ref = orc.mha_forward(*[orc.reconstruct(*orc.split_factors(as_f64(t), h)) for t in (tq, tk, tv)], bias=bias, sm_scale=scale)
    check(o, lse, o_ref, l_ref, BF16_TOL, bf16_bounds(tq, tk, tv, h, scale))
