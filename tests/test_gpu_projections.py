"""Last stage of the backward: dense gradients projected onto the rank factors.  The kernel that takes several tokens per
wave is chosen for each of q, k and v by itself."""

import numpy as np
import pytest
import torch

from conftest import make_factors
from oracle import tpa_oracle as orc
from test_gpu_backward import rel_err
from test_gpu_parity import as_f64, to_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("odd", range(6))
def test_an_unaligned_gradient_view_changes_no_other_gradient(gpu, dt, odd):
    """One gradient array starts one element past a 16-byte boundary: the other two of q, k, v stay on their kernel and so
    come out bit for bit; the pair with that array is summed in another order, which at 128 terms of either sign moves
    fp32 sums by up to 128 * 2^-24 * sqrt(128) = 8.6e-5 of the largest."""
    from tpa import tpa

    b, lq, lk, h, d = 2, 200, 331, 16, 128
    q, k, v = (to_gpu(x, dt, gpu) for x in make_factors(103, b, lq, lk, h, d, d, 6, 2, scale_by_rank=True))
    parts = [x for t in (q, k, v) for x in (t[..., :h], t[..., h:])]
    o, lse = tpa.tpa_factors(*parts, sm_scale=d**-0.5)
    do = torch.randn(o.shape, generator=torch.Generator(device=gpu).manual_seed(7), device=gpu).to(dt)

    def gradients(shifted):
        grads = []
        for i, x in enumerate(parts):
            room = torch.full((x.numel() + 4,), float("nan"), device=gpu)
            grads.append(room[i == shifted :][: x.numel()].view(x.shape))
        return tpa.tpa_factors_bwd(*parts, None, None, o, lse, do, d**-0.5, grads=grads)

    want, got = gradients(None), gradients(odd)
    assert got[odd].data_ptr() % 16 == 4
    for i, (x, y) in enumerate(zip(want, got)):
        if i // 2 != odd // 2:
            assert torch.equal(x, y), i
        else:
            assert ((x - y).abs().max() / x.abs().max()).item() <= 1e-4, i


@pytest.mark.parametrize("dt,tol", [(torch.float32, 2e-4), (torch.bfloat16, 1.5e-2)])
@pytest.mark.parametrize("dk,dv", [(64, 128), (128, 64), (64, 24), (24, 128)])
def test_head_sizes_that_differ(gpu, dt, tol, dk, dv):
    """Both head sizes on that kernel, at their own widths, or one of them; lengths of no whole workgroup."""
    from tpa import tpa

    b, lq, lk, h = 2, 37, 90, 8
    q, k, v = (to_gpu(x, dt, gpu) for x in make_factors(104, b, lq, lk, h, dk, dv, 6, 3, scale_by_rank=True))
    o, res = tpa._tpa_fwd(q, k, v, h, None, None, dk**-0.5, True, None, False, False, False)
    do = to_gpu(np.random.default_rng(9).standard_normal((b, lq, h, dv)).astype(np.float32), dt, gpu)
    got = tpa._tpa_bwd(h, dk**-0.5, True, None, False, False, False, res, do)
    want = orc.tpa_backward(as_f64(q), as_f64(k), as_f64(v), None, None, h, as_f64(do), sm_scale=dk**-0.5, causal=True)
    for name, g, w in zip("qkv", got, want):
        assert rel_err(as_f64(g), w) <= tol, name


@pytest.mark.parametrize("dt,tol", [(torch.float32, 2e-4), (torch.bfloat16, 1.5e-2)])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("h", [8, 16, 24, 32, 64])
def test_every_number_of_lanes_that_share_a_token(gpu, dt, tol, h, d):
    """One to eight groups of heads: each number of exchanges between the lanes, 24 heads (no power of two: indices by division,
    the staged projection) and 64 x 128 (more than a wave per token); token counts that end inside a wave.  Tolerances as above."""
    from tpa import tpa

    b, lq, lk = 2, 37, 91
    q, k, v = (to_gpu(x, dt, gpu) for x in make_factors(105, b, lq, lk, h, d, d, 3, 2, scale_by_rank=True))
    o, res = tpa._tpa_fwd(q, k, v, h, None, None, d**-0.5, True, None, False, False, False)
    do = to_gpu(np.random.default_rng(10).standard_normal((b, lq, h, d)).astype(np.float32), dt, gpu)
    got = tpa._tpa_bwd(h, d**-0.5, True, None, False, False, False, res, do)
    want = orc.tpa_backward(as_f64(q), as_f64(k), as_f64(v), None, None, h, as_f64(do), sm_scale=d**-0.5, causal=True)
    for name, g, w in zip("qkv", got, want):
        assert rel_err(as_f64(g), w) <= tol, name
        assert rel_err(as_f64(g)[..., :h], w[..., :h]) <= tol and rel_err(as_f64(g)[..., h:], w[..., h:]) <= tol, name
