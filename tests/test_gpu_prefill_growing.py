"""Rows whose logits grow along the keys.

The generated loops of the prefill kernel keep one reference per row and move it when the sum of a group of
exponentials says so; the group is then scaled, or, where its sum overflowed, computed again.  Here the reference has to move in every group a lane can
own (both 32-key blocks of a tile, both halves of a block, both tile parities), by little and by more than the range of a float
at once, for some rows of a wave and not for others, in both loops and both head sizes; against the emulation of the
kernels' rounding points, of which only the start of a logit's fp32 sum depends on the reference.

The head factors are powers of two on one rank, so that Q, K and V are exact before their one rounding: a rounding that falls
the other way would move a logit of a thousand by more than a group's worth."""

import numpy as np
import pytest
import torch

from error_model import LOG2E_F32, emulate_bf16_attention, reconstruct_dense, round_bf16
from test_gpu_parity import as_f64, run_bf16

pytestmark = pytest.mark.gpu


def _factors(rng, l, r, h, d):
    x = np.zeros((1, l, r, h + d))
    x[:, :, 0, :h] = r * 2.0 ** rng.integers(-1, 2, (1, l, h))  # the 1/r of the reconstruction is taken back
    x[..., h:] = round_bf16(rng.standard_normal((1, l, r, d)))
    return x


@pytest.mark.parametrize("top", [2.0, 16.0, 512.0])
@pytest.mark.parametrize("d", [128, 64])
@pytest.mark.parametrize("lq,lk,rk,causal", [(300, 1600, 2, False), (512, 1100, 4, False), (600, 600, 4, True), (300, 300, 2, True)])
def test_the_reference_moves_in_every_group(gpu, lq, lk, rk, causal, d, top):
    h, rng = 8, np.random.default_rng(91)
    scale = 0.25 * d**-0.5
    q, k, v = _factors(rng, lq, 4, h, d), _factors(rng, lk, rk, h, d), _factors(rng, lk, rk, h, d)
    # one key in 23 outgrows everything before it: the residues of its position walk through the groups
    at = np.arange(70, lk, 23)
    k[:, at, :, :h] *= 2.0 ** np.round(np.log2(top) * np.arange(1, len(at) + 1) / len(at))[None, :, None, None]
    (tq, tk, tv), o, lse = run_bf16(gpu, q, k, v, h, scale, causal)
    qd, kd, vd = (reconstruct_dense(as_f64(t), h) for t in (tq, tk, tv))
    qd = (np.float32(qd) * np.float32(np.float32(scale) * np.float32(LOG2E_F32))).astype(np.float64)  # the product in fp32, as the kernels form it
    bias = np.where(np.tril(np.ones((lq, lk), bool)), 0.0, -np.inf)[None] if causal else None
    o_e, l_e, slack = emulate_bf16_attention(qd, kd, vd, scale, bias=bias, q_prescaled=True)
    got, got_l = as_f64(o), as_f64(lse).transpose(0, 2, 1)
    assert np.isfinite(got).all() and np.isfinite(got_l).all()
    # an fp32 sum of d products: d / 16 additions into a partial sum of at most the largest |q| |k| of the row, each 2^-24 of it
    big = np.einsum("blhd->blh", np.abs(round_bf16(qd))) * np.abs(kd).max()
    noise = big * (d / 16) * 2.0**-24
    assert (np.abs(got_l - l_e) <= 2e-4 + noise).all()
    spacing = 2.0**-7 * np.maximum(np.abs(o_e), np.abs(got))
    room = 2 * noise[..., None] * np.abs(vd).max()
    assert (np.abs(got - o_e) <= 2 * spacing + slack + room).all()
    # the sums are not that far off on average: most elements are the emulation's own
    assert np.mean(np.abs(got - o_e) > spacing) <= 0.01
