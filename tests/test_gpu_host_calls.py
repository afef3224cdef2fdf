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


def _training_inputs(gpu, dt=torch.bfloat16, b=2, t=300, h=8, d=64):
    q, k, v = (to_gpu(x, dt, gpu).requires_grad_() for x in make_factors(96, b, t, t, h, d, d, 6, 2, scale_by_rank=True))
    do = torch.randn((b, t, h, d), generator=torch.Generator(device=gpu).manual_seed(3), device=gpu).to(dt)
    ids = (torch.arange(t, device=gpu, dtype=torch.int32) // 77).expand(b, t).contiguous()
    return q, k, v, do, ids


@pytest.mark.parametrize("packed", [False, True])
def test_saved_tensor_hooks_and_checkpointing(gpu, packed):
    """What the node saves goes through saved-tensor hooks (to the host and back: other storage, the same values), and a
    checkpointed call runs its forward again: the gradients are bit for bit those of the plain call."""
    from torch.utils.checkpoint import checkpoint
    from tpa import tpa

    q, k, v, do, ids = _training_inputs(gpu)
    ids = ids if packed else None
    call = lambda q, k, v: tpa.tpa(q, k, v, 8, ids, ids, sm_scale=0.125, causal=True)
    o = call(q, k, v)
    want = torch.autograd.grad(o, (q, k, v), do)
    saved = []

    def to_host(x):
        saved.append(x.shape)
        return x.detach().cpu()

    with torch.autograd.graph.saved_tensors_hooks(to_host, lambda x: x.to(gpu)):
        hooked = call(q, k, v)
    assert len(saved) == 5 and torch.equal(hooked, o)
    for x, y in zip(torch.autograd.grad(hooked, (q, k, v), do), want):
        assert torch.equal(x, y)
    for reentrant in (False, True):
        leaves = [x.detach().requires_grad_() for x in (q, k, v)]
        again = checkpoint(call, *leaves, use_reentrant=reentrant)
        again.backward(do)
        assert torch.equal(again, o)
        for x, y in zip(leaves, want):
            assert torch.equal(x.grad, y)


def test_an_input_changed_between_forward_and_backward_is_an_error(gpu):
    from tpa import tpa

    q, k, v, do, _ = _training_inputs(gpu)
    o = tpa.tpa(q, k, v, 8, sm_scale=0.125)
    with torch.no_grad():
        k.mul_(2)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        o.backward(do)


def test_calls_of_several_threads_on_streams_of_their_own(gpu):
    """Training steps and decodes of different sizes from four threads at once, each on its own stream: every result is
    that of the same call alone."""
    from concurrent.futures import ThreadPoolExecutor
    from tpa import tpa

    cases = []
    for i in range(4):
        q, k, v, do, ids = _training_inputs(gpu, t=200 + 60 * i)
        kv = [x for t in (k, v) for x in (t.detach()[..., :8].contiguous(), t.detach()[..., 8:].contiguous())]
        lengths = torch.tensor([100 + i, 200], dtype=torch.int32, device=gpu)
        last = [x.contiguous() for x in (q.detach()[:, -1:, :, :8], q.detach()[:, -1:, :, 8:])]
        cases.append((q, k, v, do, ids, last, kv, lengths))

    def step(case):
        q, k, v, do, ids, last, kv, lengths = case
        o = tpa.tpa(q, k, v, 8, ids, ids, sm_scale=0.125, causal=True)
        return (o.detach(), *torch.autograd.grad(o, (q, k, v), do), *tpa.tpa_decode(*last, *kv, sm_scale=0.125, kv_lengths=lengths))

    want = [step(c) for c in cases]
    torch.cuda.synchronize()

    def worker(case):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            for _ in range(10):
                got = step(case)
        stream.synchronize()
        return got

    with ThreadPoolExecutor(4) as pool:
        for got, alone in zip(pool.map(worker, cases), want):
            for x, y in zip(got, alone):
                assert torch.equal(x, y)
