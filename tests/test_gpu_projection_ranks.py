"""Short calls, whose ranks are projected by workgroups of their own: gradients of every rank against the oracle."""

import numpy as np
import pytest
import torch

from conftest import make_factors
from oracle import tpa_oracle as orc
from test_gpu_backward import rel_err
from test_gpu_parity import as_f64, to_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt,tol", [(torch.float32, 2e-4), (torch.bfloat16, 1.5e-2)])
@pytest.mark.parametrize(
    "b,lq,lk,h,d,rq,rk",
    [
        (1, 70, 33, 8, 64, 6, 2),     # two ranks each
        (2, 40, 90, 8, 128, 16, 8),
        (1, 65, 64, 16, 64, 7, 3),    # a last workgroup with one rank
        (3, 64, 150, 8, 64, 2, 11),   # most of them on the other side
        (1, 80, 80, 8, 64, 1, 1),     # nothing to deal
        (1, 64, 64, 16, 128, 33, 1),  # more ranks than parts
        (1, 700, 300, 16, 64, 16, 8),  # 400 workgroups or fewer only with eight ranks each
        (1, 1600, 1600, 8, 64, 16, 8),
        (1, 96, 64, 8, 256, 5, 2),    # the other kernel
        (1, 400, 400, 16, 64, 6, 4),  # two ranks each, 25 workgroups in 32
        (3, 300, 17, 16, 64, 6, 4),   # 19 in 24, one of them with keys
        (1, 512, 400, 8, 128, 4, 3),  # 32
    ],
)
def test_gradients_of_every_rank(gpu, dt, tol, b, lq, lk, h, d, rq, rk):
    from tpa import tpa

    if rq == rk == 1:
        # Q and K of one rank are products of two normal numbers: logits reach a_q a_k |b_q| |b_k| / sqrt(d) = 3 * 3 * 3, and operands
        # rounded to 8 bits move a weight by up to 27 * 2^-8 = 0.1 of itself.  fp32 operands: 27 * 2^-23, within its tolerance
        dt, tol = torch.float32, 2e-4
    q, k, v = (to_gpu(x, dt, gpu) for x in make_factors(lq + rq, b, lq, lk, h, d, d, rq, rk, scale_by_rank=True))
    o, res = tpa._tpa_fwd(q, k, v, h, None, None, d**-0.5, False, None, False, False, False)
    do = to_gpu(np.random.default_rng(9).standard_normal((b, lq, h, d)).astype(np.float32), dt, gpu)
    got = tpa._tpa_bwd(h, d**-0.5, False, None, False, False, False, res, do)
    want = orc.tpa_backward(as_f64(q), as_f64(k), as_f64(v), None, None, h, as_f64(do), sm_scale=d**-0.5, causal=False)
    for name, g, w in zip("qkv", got, want):
        assert rel_err(as_f64(g), w) <= tol, name


@pytest.mark.parametrize("odd", range(6))
def test_one_array_on_the_other_kernel(gpu, odd):
    """At a length at which the ranks are dealt, with one array that is not aligned: two arrays remain in the launch."""
    from tpa import tpa

    b, lq, lk, h, d = 1, 90, 70, 8, 64
    q, k, v = (to_gpu(x, torch.float32, gpu) for x in make_factors(103, b, lq, lk, h, d, d, 6, 4, scale_by_rank=True))
    parts = [x for t in (q, k, v) for x in (t[..., :h], t[..., h:])]
    o, lse = tpa.tpa_factors(*parts, sm_scale=d**-0.5)
    do = torch.randn(o.shape, generator=torch.Generator(device=gpu).manual_seed(7), device=gpu)

    def gradients(shifted):
        grads = []
        for i, x in enumerate(parts):
            room = torch.full((x.numel() + 4,), float("nan"), device=gpu)
            grads.append(room[i == shifted :][: x.numel()].view(x.shape))
        return tpa.tpa_factors_bwd(*parts, None, None, o, lse, do, d**-0.5, grads=grads)

    want, got = gradients(None), gradients(odd)
    for i, (x, y) in enumerate(zip(want, got)):
        if i // 2 != odd // 2:
            assert torch.equal(x, y), i
        else:  # fp32 sums of 64 terms in another order
            assert ((x - y).abs().max() / x.abs().max()).item() <= 1e-4, i
