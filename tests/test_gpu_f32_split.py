"""fp32 attention, forward and backward, on the bf16 matrix cores (products of three-way splits): values that do not split - infinities, NaN, numbers
that round up to infinity in bf16, numbers whose parts would be denormal - in each of the workgroup forms, against float64.

Tolerance: the kernels' own error on ordinary values is below 1e-6 of the result's norm; 1e-5 leaves ten times that, and
a part lost from a split (2^-8 or 2^-16 of a value) exceeds it.
"""

import numpy as np
import pytest
import torch

from conftest import make_factors
from oracle import tpa_oracle as orc

pytestmark = pytest.mark.gpu

SHAPES = [
    (1, 70, 2, 64, 2),     # 32 rows, waves split the keys, rank 2
    (1, 290, 2, 64, 1),    # rank 1
    (1, 70, 2, 128, 3),    # head size 128, any rank
    (1, 300, 64, 64, 2),   # 192 workgroups of 128 rows
    (2, 300, 64, 64, 2),   # 256 rows
    (2, 300, 64, 128, 2),
]


def _spoil(kind, q, k, v, h):
    """Puts values that do not split into the factors (head factors first in the last dimension)."""
    key = 5
    if kind == "infinite key":  # logit -inf for every row: the key drops out
        q[:, :, :, :h] = np.abs(q[:, :, :, :h])
        q[:, :, :, h] = np.abs(q[:, :, :, h])
        k[:, key, :, :h] = np.abs(k[:, key, :, :h])
        k[:, key, 0, h] = -np.inf
    elif kind == "infinite query":  # head-independent -inf logits against keys with a negative first component
        q[:, 3, :, :h] = np.abs(q[:, 3, :, :h])
        q[:, 3, 0, h] = np.inf
        k[:, :, :, :h] = np.abs(k[:, :, :, :h])
        k[:, :, :, h] = -np.abs(k[:, :, :, h])
        k[:, key, :, h] = 0.0  # inf * 0: this row is NaN
    elif kind == "NaN value":  # spoils one column of the result and no other
        v[:, key, 0, h + 7] = np.nan
    elif kind == "infinite value":
        v[:, key, :, :h] = np.abs(v[:, key, :, :h])
        v[:, key, 0, h + 7] = np.inf
    elif kind == "rounds to infinity":  # finite, but its bf16 neighbour is not
        v[:, :, :, :h] = 1.0
        v[:, key, :, h + 7] = 3.3985e38
        v[:, key, 1:, h + 7] = 0.0
    elif kind == "tiny values":
        v[:, :, :, h:] *= 1e-33
    elif kind == "one small column":  # below 2^-110, where the last bits of a value are below bf16's smallest number
        v[:, :, :, h + 6] *= 2e-37
    elif kind == "one small column beside an infinity":
        v[:, :, :, h + 6] *= 2e-37
        v[:, key, :, :h] = np.abs(v[:, key, :, :h])
        v[:, key, 0, h + 7] = np.inf
    elif kind == "small queries, large keys":  # products around 1 of parts whose last bits are below bf16's smallest number
        q[:, :, :, h:] *= 1e-35
        k[:, :, :, h:] *= 1e35
    elif kind == "logit below the range":  # finite operands, products around -2^140 of which the parts have both signs
        q[:, :, :, :h] = np.abs(q[:, :, :, :h]) + 0.5
        k[:, key, :, :h] = np.abs(k[:, key, :, :h]) + 0.5
        q[:, :, :, h] = np.float32(1.302 * 2.0**70)
        k[:, :, :, h] = 0.0
        k[:, key, :, h] = np.float32(-1.302 * 2.0**70)
    elif kind == "tiny queries, large keys":
        q[:, :, :, h:] *= 1e-19
        k[:, :, :, h:] *= 1e19


@pytest.mark.parametrize("kind", ["ordinary", "infinite key", "infinite query", "NaN value", "infinite value", "rounds to infinity", "tiny values", "tiny queries, large keys", "logit below the range", "one small column", "one small column beside an infinity", "small queries, large keys"])
@pytest.mark.parametrize("b,t,h,d,rk", SHAPES)
def test_forward_values_that_do_not_split(gpu, b, t, h, d, rk, kind):
    from tpa import tpa

    q, k, v = make_factors(81, b, t, t, h, d, d, 3, rk, scale_by_rank=True)
    _spoil(kind, q, k, v, h)
    scale = d**-0.5
    sp = lambda x: (torch.from_numpy(x[..., :h].copy()).to(gpu), torch.from_numpy(x[..., h:].copy()).to(gpu))
    o, _ = tpa.tpa_factors(*sp(q), *sp(k), *sp(v), None, None, scale, False, kernel=2)
    with np.errstate(all="ignore"):
        want, _ = orc.tpa_reference(q.astype(np.float64), k.astype(np.float64), v.astype(np.float64), None, None, h, sm_scale=scale)
    got = o.cpu().numpy().astype(np.float64)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(np.isposinf(got), np.isposinf(want))
    ok = np.isfinite(want)
    assert ok.mean() > 0.9
    # column by column: a column of small values has to be as accurate as the others
    for c in range(d):
        m = ok[..., c]
        x, y = got[..., c][m], want[..., c][m]
        if x.size:
            top = np.abs(y).max()
            assert np.linalg.norm((x - y) / top) <= 1e-5 * np.linalg.norm(y / top), c


@pytest.mark.parametrize("kind", ["ordinary", "small gradient", "tiny gradient", "one tiny column", "rounds to infinity", "large gradient"])
@pytest.mark.parametrize(
    "b,t,h,d,causal",
    [
        (1, 70, 2, 64, True),     # 32 rows, waves split the streamed tiles
        (1, 70, 2, 128, False),
        (1, 300, 64, 64, False),  # 192 blocks of 128 rows, four waves
        (2, 300, 64, 64, False),  # 256 blocks of 256 rows, eight waves
        (4, 390, 64, 64, True),   # 512 of them, causal
        (2, 300, 32, 128, False),
    ],
)
def test_backward_values_that_do_not_split(gpu, b, t, h, d, causal, kind):
    from tpa import tpa

    q, k, v = make_factors(83, b, t, t, h, d, d, 2, 2, scale_by_rank=True)
    do = np.random.default_rng(84).standard_normal((b, t, h, d)).astype(np.float32)
    if kind == "tiny gradient":
        do *= np.float32(1e-28)
    elif kind == "small gradient":  # small, but split
        do *= np.float32(1e-20)
    elif kind == "one tiny column":  # of the upstream gradient and of the values
        do[..., 6] *= np.float32(2e-37)
        v[..., h + 7] *= np.float32(2e-37)
    elif kind == "large gradient":  # dP and dS near the largest float
        do *= np.float32(1e16)
        v[..., h:] *= np.float32(1e20)
    elif kind == "rounds to infinity":
        _spoil(kind, q, k, v, h)
        do[..., 7] *= np.float32(1e-30)
    scale = d**-0.5
    sp = lambda x: (torch.from_numpy(x[..., :h].copy()).to(gpu), torch.from_numpy(x[..., h:].copy()).to(gpu))
    o, lse = tpa.tpa_factors(*sp(q), *sp(k), *sp(v), None, None, scale, causal, kernel=2)
    grads = tpa.tpa_factors_bwd(*sp(q), *sp(k), *sp(v), None, None, o, lse, torch.from_numpy(do).to(gpu), scale, causal, kernel=2)
    want = orc.tpa_backward(q, k, v, None, None, h, do, sm_scale=scale, causal=causal)
    for n, w in enumerate(want):
        got = np.concatenate([x.cpu().numpy() for x in grads[2 * n : 2 * n + 2]], axis=-1).astype(np.float64)
        # the head factors' gradients as a whole, the token factors' column by column
        for x, y in [(got[..., :h], w[..., :h])] + [(got[..., h + c], w[..., h + c]) for c in range(d)]:
            top = np.abs(y).max()
            assert np.linalg.norm((x - y) / top) <= 1e-5 * np.linalg.norm(y / top), "qkv"[n]
