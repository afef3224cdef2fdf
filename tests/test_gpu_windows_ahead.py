"""Packed documents: the windows of ids that the launch of the dense arrays finds for the attention kernels, under every mask they
take into account - blocks of rows with a last one of a single row, ids in and out of order, lengths and offsets - and on either side of the
4096 (forward) and 8192 (backward) tokens times (batch, head) pairs from which they are found there.

Forward: the route over dense tiles against the fused kernel, which scans the ids itself, on factors whose Q, K and V are exact; the
tolerance is that of test_gpu_prefill_four_waves.py.  Backward: against the oracle.  A row's dS is a difference, p (dP - delta), of terms
rounded to 2^-8 (dP's operands once each, the output inside delta, dS itself), and where documents leave a row few keys the terms are
up to twice as large as what is left of them: 2 x 4 x 2^-8 of the largest gradient.  A key that is not visited is off by its whole weight."""

import numpy as np
import pytest
import torch

from conftest import make_factors, segment_ids
from oracle import tpa_oracle as orc
from test_gpu_backward import rel_err
from test_gpu_parity import as_f64, to_gpu

pytestmark = pytest.mark.gpu


def _ids(kind, b, lq, lk, rng):
    if kind == "in no order":
        return tuple(rng.integers(0, 4, (b, n)).astype(np.int32) for n in (lq, lk))
    ids = segment_ids(max(lq, lk), 97, b)
    if kind == "falling":
        ids = ids.max() - ids
    return ids[:, :lq].copy(), ids[:, :lk].copy()


@pytest.mark.parametrize("kind", ["documents", "falling", "in no order"])
@pytest.mark.parametrize("mask", ["none", "causal", "offset", "behind", "lengths", "bottom right"])
@pytest.mark.parametrize("b,h,d,lq,lk", [(2, 8, 64, 385, 385), (1, 24, 64, 641, 1100), (3, 8, 128, 257, 700), (2, 8, 128, 513, 300), (1, 8, 64, 511, 500), (1, 8, 64, 300, 512)])
def test_forward(gpu, b, h, d, lq, lk, mask, kind):
    from tpa import tpa

    gen = torch.Generator(device="cpu").manual_seed(lq)

    def make(l):
        x = torch.zeros((b, l, 4, h + d))
        x[:, :, 0, :h] = 4 * 2.0 ** torch.randint(-1, 2, (b, l, h), generator=gen)
        x[..., h:] = torch.randn((b, l, 4, d), generator=gen)
        return x.to(torch.bfloat16).to(gpu)

    args = [p for x in (make(lq), make(lk), make(lk)) for p in (x[..., :h], x[..., h:])]
    kw = dict(sm_scale=d**-0.5, causal=mask in ("causal", "offset", "behind"), kernel=2)
    kw["causal_offset"] = {"offset": 130, "behind": -70}.get(mask, 0)
    if mask == "bottom right":
        kw["causal"] = tpa.CAUSAL_BOTTOM_RIGHT
    if mask in ("lengths", "bottom right"):
        kw["kv_lengths"] = torch.tensor([lk, lk - 77, 0][:b], dtype=torch.int32, device=gpu)
    q_ids, k_ids = (torch.from_numpy(x).to(gpu) for x in _ids(kind, b, lq, lk, np.random.default_rng(lk)))
    (o1, l1), (o2, l2) = (tpa.tpa_factors(*args, q_ids, k_ids, use_workspace=w, **kw) for w in (True, False))
    x, y = (o.float().cpu().numpy().astype(np.float64) for o in (o1, o2))
    np.testing.assert_array_equal(np.isnan(x), np.isnan(y))
    slack = np.maximum(2.0**-7 * np.abs(y), 2.0**-8 * np.max(np.abs(np.nan_to_num(y)), axis=-1, keepdims=True))
    assert not (np.abs(x - y) > slack).any()
    a, c = (l.cpu().numpy() for l in (l1, l2))
    seen = np.isfinite(c)
    np.testing.assert_array_equal(np.isfinite(a), seen)
    assert np.abs(a[seen] - c[seen]).max(initial=0.0) <= 1e-5


@pytest.mark.parametrize("kind", ["documents", "falling", "in no order"])
@pytest.mark.parametrize("causal,offset", [(False, 0), (True, 0), (True, 70)])
@pytest.mark.parametrize("b,h,d,lq,lk", [(2, 8, 64, 129, 129), (1, 16, 64, 300, 257), (2, 8, 128, 257, 300), (2, 16, 128, 257, 300), (2, 16, 64, 300, 257), (2, 8, 64, 130, 512)])
def test_backward(gpu, b, h, d, lq, lk, causal, offset, kind):
    from tpa import tpa

    q, k, v = (to_gpu(x, torch.bfloat16, gpu) for x in make_factors(117, b, lq, lk, h, d, d, 3, 2, scale_by_rank=True))
    q_ids, k_ids = _ids(kind, b, lq, lk, np.random.default_rng(lk))
    k_ids[:, 0] = q_ids[:, 0]
    tq, tk = (torch.from_numpy(x).to(gpu) for x in (q_ids, k_ids))
    args = [p for x in (q, k, v) for p in (x[..., :h], x[..., h:])]
    kw = dict(sm_scale=d**-0.5, causal=causal, causal_offset=offset, kernel=2)
    o, lse = tpa.tpa_factors(*args, tq, tk, **kw)
    do = to_gpu(np.random.default_rng(12).standard_normal((b, lq, h, d)).astype(np.float32), torch.bfloat16, gpu)
    grads = tpa.tpa_factors_bwd(*args, tq, tk, o, lse, do, **kw)
    bias = np.where(q_ids[:, :, None] == k_ids[:, None, :], 0.0, -np.inf)
    if causal:
        bias = np.where(np.tril(np.ones((lq, lk), bool), k=offset), bias, -np.inf)
    want = _oracle_gradients(q, k, v, h, bias, as_f64(do), d**-0.5)
    for n in range(0, 6, 2):  # of the largest entry of either factor's gradient, as the concatenated gradients of the other tests
        assert rel_err(np.concatenate([as_f64(g) for g in grads[n : n + 2]], -1), np.concatenate(want[n : n + 2], -1)) <= 2.0**-5, n


def _oracle_gradients(q, k, v, h, bias, do, scale):
    factors = [orc.split_factors(as_f64(t), h) for t in (q, k, v)]
    dense = [orc.reconstruct(*f) for f in factors]
    grads = orc.mha_backward(*dense, bias, scale, do)
    return [x for g, f in zip(grads, factors) for x in orc.project_to_factors(g, *f)]
