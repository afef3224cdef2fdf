"""The native host layer (csrc/host_calls.cc) on the GPU: what torch programs do around a call."""

import pytest
import torch

from conftest import make_factors
from test_gpu_parity import to_gpu

pytestmark = pytest.mark.gpu


def test_a_card_too_full_for_the_optional_workspace(gpu):
    """256 rows over 16384 keys at rank 4 ask for 270 MB of dense keys and values; where they do not fit, the kernel that takes
    none serves the call: the result is bit for bit that of `use_workspace=False`."""
    from tpa import tpa

    h, d = 32, 128
    q, k, v = (to_gpu(x, torch.bfloat16, gpu) for x in make_factors(95, 1, 256, 16384, h, d, d, 2, 4, scale_by_rank=True))
    parts = [x for t in (q, k, v) for x in (t[..., :h], t[..., h:])]
    want, want_lse = tpa.tpa_factors(*parts, sm_scale=d**-0.5, use_workspace=False)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(gpu).total_memory
    try:
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved(gpu) + (64 << 20)) / total, gpu)
        got, got_lse = tpa.tpa_factors(*parts, sm_scale=d**-0.5)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0, gpu)
    assert torch.equal(got, want) and torch.equal(got_lse, want_lse)
