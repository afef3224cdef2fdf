"""Query rows of NaN in the generated loops of the prefill kernel: they end as NaN and leave every other row to its own
result, also where a row of the same wave moves its reference in the same groups."""

import numpy as np
import pytest
import torch

from conftest import make_factors
from test_gpu_parity import run_bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [128, 64])
@pytest.mark.parametrize("lq,lk,rk,causal", [(300, 1600, 2, False), (512, 1100, 4, False), (600, 600, 4, True), (300, 300, 2, True)])
def test_a_row_of_nan_leaves_the_others_alone(gpu, lq, lk, rk, causal, d):
    h = 8
    q, k, v = make_factors(71, 1, lq, lk, h, d, d, 4, rk, scale_by_rank=True)
    k[:, 70::23, :, :h] *= np.linspace(1.0, 400.0, len(range(70, lk, 23)))[None, :, None, None]  # the reference moves
    _, o, lse = run_bf16(gpu, q, k, v, h, d**-0.5, causal)
    dead = np.arange(5, lq, 37)
    q[:, dead] = np.nan
    _, o_nan, lse_nan = run_bf16(gpu, q, k, v, h, d**-0.5, causal)
    alive = np.setdiff1d(np.arange(lq), dead)
    assert torch.isnan(o_nan[:, dead]).all()
    # The rows of a wave move their references together, so that a row's may move at another tile without its neighbours.  An
    # fp32 sum of d products that starts elsewhere is off by d / 16 roundings of at most 2^-24 of its size (logits below 2^12:
    # 2^-9); a probability may then fall to its neighbour in bf16, 2^-8 of it, and so may the result, 2^-8 of that.
    assert (lse_nan[:, :, alive] - lse[:, :, alive]).abs().max().item() <= 2.0**-9
    big = float(np.abs(v[..., h:]).max() * np.abs(v[..., :h]).max())
    assert (o_nan[:, alive].float() - o[:, alive].float()).abs().max().item() <= (2.0**-8 + 2.0**-8) * big
