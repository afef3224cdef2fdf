"""Packed sequences: the scan for the first and the last element that a workgroup's ids can meet, on rows of ids that begin at
every offset from a 16-byte boundary and are longer than one pass of the largest workgroup."""

import numpy as np
import pytest
import torch

from conftest import make_factors
from oracle import tpa_oracle as orc
from test_gpu_backward import rel_err
from test_gpu_parity import as_f64, to_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt,tol", [(torch.float32, 2e-4), (torch.bfloat16, 1.5e-2)])
@pytest.mark.parametrize("n", [5, 8202, 8203, 8205])
@pytest.mark.parametrize("rows_are_long", [False, True])
@pytest.mark.parametrize("at", [(0, -1), (1, -2), (2, -1), (0, -3), (3, 7)])
def test_two_matching_elements_at_the_ends_of_the_row(gpu, dt, tol, n, rows_are_long, at):
    """Only the elements `at` of the long side carry the short side's id: one of them missed, and a row of the softmax loses a
    key (half of its output or so) or a key its gradient.  Tolerances as in the other tests of the gradients; the
    forward is held to the same share of its largest value."""
    from tpa import tpa

    b, m, h, d = 3, 40, 8, 64
    lq, lk = (n, m) if rows_are_long else (m, n)
    q, k, v = (to_gpu(x, dt, gpu) for x in make_factors(111, b, lq, lk, h, d, d, 3, 2, scale_by_rank=True))
    ids = np.full((b, n), 1, np.int32)
    ids[:, [x % n for x in at]] = 7
    short = np.full((b, m), 7, np.int32)
    qseg, kvseg = (ids, short) if rows_are_long else (short, ids)
    tqs, tks = torch.from_numpy(qseg).to(gpu), torch.from_numpy(kvseg).to(gpu)
    o, res = tpa._tpa_fwd(q, k, v, h, tqs, tks, d**-0.5, False, None, False, False, False)
    visible = qseg[0] == 7
    o_ref, _ = orc.tpa_reference(as_f64(q), as_f64(k), as_f64(v), qseg, kvseg, h, sm_scale=d**-0.5)
    assert rel_err(as_f64(o)[:, visible], np.asarray(o_ref)[:, visible]) <= tol
    do = to_gpu(np.random.default_rng(12).standard_normal((b, lq, h, d)).astype(np.float32), dt, gpu)
    got = tpa._tpa_bwd(h, d**-0.5, False, None, False, False, False, res, do)
    want = orc.tpa_backward(as_f64(q), as_f64(k), as_f64(v), qseg, kvseg, h, as_f64(do), sm_scale=d**-0.5, causal=False)
    for name, g, w in zip("qkv", got, want):
        assert rel_err(as_f64(g), w) <= tol, name
