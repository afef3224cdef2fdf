"""Workgroups of four waves at head size 64 against kernels of eight - dense tiles against the any-rank fused kernel, the rank-2 fused
kernel against the any-rank one through a zero third rank: rows around a workgroup's
128, too few tiles for the pipelined loop and many, every mask; and the generated loop against its asm statement.

Tolerance: both round at the same places, but a logit's fp32 sum starts at the row's reference, which the two move at different
keys, so that a probability may round to the neighbouring bf16 value: at most 2^-8 of the largest value it weighs (few of them
do; the row's largest result stands for it, as rows whose few keys weigh that much have), and the result itself 2^-7 of its
magnitude.  The logsumexp is fp32 and says sharply which keys were seen: 1e-5 where one key of 1500 is 7e-4."""

import numpy as np
import pytest
import torch

from conftest import segment_ids
from test_prefill_loop_generator import test_generated_loop_matches_its_asm_statement as check_loop


@pytest.mark.parametrize("loader", ["dense4w", "r24w"])
def test_generated_loop(tmp_path, loader):
    check_loop(tmp_path, 64, loader)


MASKS = ["none", "causal", "offset", "bottom right", "lengths", "packed", "one document", "ids in no order", "no common id"]
SHAPES = [(1, 8, 257, 257), (2, 16, 383, 1100), (3, 8, 640, 321), (1, 8, 1023, 1500), (5, 64, 385, 385), (4, 16, 1409, 1409)]


@pytest.mark.gpu
@pytest.mark.parametrize("mask", MASKS)
@pytest.mark.parametrize("b,h,lq,lk", SHAPES)
def test_dense_tiles(gpu, b, h, lq, lk, mask):
    _compare(gpu, b, h, lq, lk, mask, 4)


@pytest.mark.gpu
@pytest.mark.parametrize("mask", MASKS)
@pytest.mark.parametrize("b,h,lq,lk", [(1, 8, 17, 300), (1, 8, 127, 127), (2, 24, 129, 70)] + SHAPES[:-1])
def test_rank_two_fused(gpu, b, h, lq, lk, mask):
    _compare(gpu, b, h, lq, lk, mask, 2)


def _compare(gpu, b, h, lq, lk, mask, rk):
    from tpa import tpa

    d = 64
    gen = torch.Generator(device="cpu").manual_seed(lq)

    def make(l, r):  # head factors that are powers of two on one rank: Q, K and V are exact, whatever order sums the ranks
        x = torch.zeros((b, l, r, h + d))
        x[:, :, 0, :h] = r * 2.0 ** torch.randint(-1, 2, (b, l, h), generator=gen)
        x[..., h:] = torch.randn((b, l, r, d), generator=gen)
        return x.to(torch.bfloat16).to(gpu)

    q, k, v = make(lq, 4), make(lk, rk), make(lk, rk)
    args = [p for x in (q, k, v) for p in (x[..., :h], x[..., h:])]
    kw = dict(sm_scale=d**-0.5, causal=mask in ("causal", "offset", "packed", "one document"), kernel=2)
    if mask == "offset":
        kw["causal_offset"] = lk - lq
    if mask == "bottom right":
        kw["causal"] = tpa.CAUSAL_BOTTOM_RIGHT
    if mask in ("lengths", "bottom right"):
        kw["kv_lengths"] = torch.tensor([max(0, lk - 77 * i * i) for i in range(b)], dtype=torch.int32, device=gpu)
    if mask in ("packed", "one document"):
        longest = max(lq, lk)
        ids = torch.from_numpy(segment_ids(longest, 97 if mask == "packed" else longest, b)).to(gpu)
        kw["q_segment_ids"], kw["kv_segment_ids"] = ids[:, :lq].contiguous(), ids[:, :lk].contiguous()
    if mask in ("ids in no order", "no common id"):
        kw["q_segment_ids"] = torch.randint(0, 3, (b, lq), generator=gen, dtype=torch.int32).to(gpu)
        kw["kv_segment_ids"] = torch.randint(0, 3, (b, lk), generator=gen, dtype=torch.int32).to(gpu) + (5 if mask == "no common id" else 0)
    o1, l1 = tpa.tpa_factors(*args, use_workspace=rk != 2, **kw)
    if rk == 2:  # a third rank of zeros and half as much again on the others: the same K and V (three is no power of two, 1.5 is exact)
        for n in range(2, 6):
            args[n] = torch.cat([args[n] * 1.5 if n % 2 == 0 else args[n], torch.zeros_like(args[n][:, :, :1])], 2)
    o2, l2 = tpa.tpa_factors(*args, use_workspace=False, **kw)
    x, y = (o.float().cpu().numpy().astype(np.float64) for o in (o1, o2))
    np.testing.assert_array_equal(np.isnan(x), np.isnan(y))
    if mask != "no common id":
        slack = np.maximum(2.0**-7 * np.abs(y), 2.0**-8 * np.nanmax(np.abs(y), axis=-1, keepdims=True, initial=0.0))
        assert not (np.abs(x - y) > slack).any()
    a, c = (l.cpu().numpy() for l in (l1, l2))
    seen = np.isfinite(c)
    np.testing.assert_array_equal(np.isfinite(a), seen)
    assert np.abs(a[seen] - c[seen]).max(initial=0.0) <= 1e-5
