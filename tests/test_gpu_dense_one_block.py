"""bf16 forward of one block of query rows over fewer than 1024 keys through dense Q, K and V: which calls ask for the room (no GPU needed),
and that the route agrees with the kernels that rebuild every tile from the factors, over masks, strides and lengths around the tiles."""

import ctypes

import numpy as np
import pytest
import torch

from conftest import segment_ids
from test_abi import _forward_call


@pytest.mark.parametrize(
    "B,H,D,lq,lk,rk,dense",
    [
        (1, 8, 64, 17, 64, 4, False),
        (1, 8, 64, 250, 250, 4, True),
        (1, 8, 64, 250, 250, 1, False),
        (1, 8, 64, 250, 900, 1, True),
        (8, 64, 64, 200, 200, 4, False),
        (8, 64, 64, 200, 200, 8, True),
        (8, 32, 128, 250, 250, 1, False),
        (8, 32, 128, 250, 1023, 4, True),
        (1, 16, 128, 250, 1023, 2, False),  # rank 2 has a rebuild of its own
        (1, 20, 128, 250, 900, 8, False),   # heads in no groups of eight
    ],
)
def test_which_calls_ask_for_it(B, H, D, lq, lk, rk, dense):
    from tpa import _dispatch as d

    lib = d.load_library()
    fake = d.TpaFactor(256, 8, 8, 8)
    call = _forward_call(B=B, H=H, D=D, lq=lq, lk=lk, rk=rk, qa=fake, qb=fake, ka=fake, kb=fake, va=fake, vb=fake)
    call.kernel = d.KERNEL_MFMA
    call.num_splits = 1
    need = lib.tpa_fwd_call_workspace_bytes(ctypes.byref(call))
    slot = lambda n: (2 * n + 255) // 256 * 256
    assert need == (slot(B * lq * H * D) + 2 * slot(B * lk * H * D) if dense else 0)
    assert need <= lib.tpa_fwd_best_workspace_bytes(B, lq, lk, H, D, D, 6, rk)
    call.ka = d.TpaFactor(256, 8, 4, 8)  # rows of head factors that start between 16 bytes: three launches, not worth it here
    assert lib.tpa_fwd_call_workspace_bytes(ctypes.byref(call)) == 0


@pytest.mark.parametrize(
    "B,H,D,lq,lk,rq,rk,dense",
    [
        (5, 32, 128, 125, 125, 6, 4, True),
        (5, 32, 128, 125, 125, 2, 4, False),  # Q of few ranks is soon summed
        (10, 8, 128, 217, 458, 6, 1, True),
        (10, 8, 128, 217, 458, 2, 1, False),
        (10, 8, 128, 217, 458, 2, 4, True),
        (4, 8, 128, 79, 79, 4, 3, True),
        (1, 8, 64, 250, 250, 2, 4, True),
        (1, 8, 128, 200, 600, 6, 2, True),
        (1, 8, 128, 200, 600, 5, 2, False),
    ],
)
def test_ranks_of_q(B, H, D, lq, lk, rq, rk, dense):
    from tpa import _dispatch as d

    lib = d.load_library()
    fake = d.TpaFactor(256, 8, 8, 8)
    call = _forward_call(B=B, H=H, D=D, lq=lq, lk=lk, rk=rk, rq=rq, qa=fake, qb=fake, ka=fake, kb=fake, va=fake, vb=fake, num_splits=1)
    slot = lambda n: (2 * n + 255) // 256 * 256
    assert lib.tpa_fwd_call_workspace_bytes(ctypes.byref(call)) == (slot(B * lq * H * D) + 2 * slot(B * lk * H * D) if dense else 0)


@pytest.mark.parametrize(
    "B,H,D,lq,lk,rq,rk,mask,dense",
    [
        (11, 16, 128, 47, 882, 2, 3, dict(), True),
        (11, 16, 128, 47, 882, 2, 3, dict(causal=1), False),                       # one tile in reach of 14
        (11, 16, 128, 47, 882, 16, 3, dict(causal=1), True),                       # but many ranks of Q
        (11, 16, 128, 47, 882, 2, 3, dict(causal=1, causal_offset=835), True),
        (11, 16, 128, 47, 882, 16, 3, dict(causal=1, causal_offset=-47), False),   # none
        (4, 64, 64, 95, 867, 2, 3, dict(), True),
        (4, 64, 64, 95, 867, 2, 3, dict(q_segment_ids=256, kv_segment_ids=256), False),   # documents: nine of 14 tiles met
        (1, 8, 64, 250, 900, 6, 4, dict(q_segment_ids=256, kv_segment_ids=256), True),
        (1, 16, 128, 33, 1100, 6, 4, dict(causal=1), True),                        # as long as that the lengths decide
    ],
)
def test_keys_that_no_row_meets_do_not_count(B, H, D, lq, lk, rq, rk, mask, dense):
    from tpa import _dispatch as d

    lib = d.load_library()
    fake = d.TpaFactor(256, 8, 8, 8)
    call = _forward_call(B=B, H=H, D=D, lq=lq, lk=lk, rq=rq, rk=rk, qa=fake, qb=fake, ka=fake, kb=fake, va=fake, vb=fake, num_splits=1, **mask)
    slot = lambda n: (2 * n + 255) // 256 * 256
    assert lib.tpa_fwd_call_workspace_bytes(ctypes.byref(call)) == (slot(B * lq * H * D) + 2 * slot(B * lk * H * D) if dense else 0)


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["concatenated", "split", "ranks first", "head factors apart"])
@pytest.mark.parametrize("mask", ["none", "causal", "offset", "bottom right", "lengths", "packed", "ids in no order", "no common id"])
@pytest.mark.parametrize("b,h,d,lq,lk,rk", [(1, 8, 64, 256, 256, 4), (2, 16, 64, 1, 1023, 8), (3, 8, 128, 33, 129, 5), (2, 40, 128, 129, 700, 3), (1, 8, 64, 130, 900, 1)])
def test_both_routes_agree(gpu, b, h, d, lq, lk, rk, mask, layout):
    """Each route rounds Q, K, V, the probabilities and the result to 8 bits, so that either is within 2^-7 of the largest value of the
    result in fp32, and they are within twice that of each other; the logarithms stay in fp32, of logits whose operands are rounded."""
    from tpa import tpa

    gen = torch.Generator(device="cpu").manual_seed(lk)

    def factors(l, r):
        x = (torch.randn((b, l, r, h + d), generator=gen) / r**0.5).to(gpu, torch.bfloat16)
        parts = x[..., :h], x[..., h:]
        if layout == "split":
            return tuple(p.contiguous() for p in parts)
        if layout == "ranks first":
            return tuple(p.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3) for p in parts)
        if layout == "head factors apart":  # rows of h + 3 elements: the route that rebuilds takes them, with or without the room
            return torch.nn.functional.pad(parts[0], (0, 3))[..., :h], parts[1]
        return parts

    args = list(factors(lq, 6) + factors(lk, rk) + factors(lk, rk))
    kw = dict(sm_scale=d**-0.5, causal=mask in ("causal", "offset", "packed"), kernel=2)
    if mask == "offset":
        kw["causal_offset"] = lk - lq
    if mask == "bottom right":
        kw["causal"] = tpa.CAUSAL_BOTTOM_RIGHT
    if mask in ("lengths", "bottom right"):
        kw["kv_lengths"] = torch.tensor([lk - 63 * i for i in range(b)], dtype=torch.int32, device=gpu)
    if mask == "packed":
        ids = torch.from_numpy(segment_ids(max(lq, lk), 97, b)).to(gpu)
        kw["q_segment_ids"], kw["kv_segment_ids"] = ids[:, :lq].contiguous(), ids[:, :lk].contiguous()
    if mask in ("ids in no order", "no common id"):
        kw["q_segment_ids"] = torch.randint(0, 3, (b, lq), generator=gen, dtype=torch.int32).to(gpu)
        kw["kv_segment_ids"] = torch.randint(0, 3, (b, lk), generator=gen, dtype=torch.int32).to(gpu) + (5 if mask == "no common id" else 0)
    (o1, l1), (o2, l2) = (tpa.tpa_factors(*args, use_workspace=w, **kw) for w in (True, False))
    x, y = (o.float().cpu().numpy().astype(np.float64) for o in (o1, o2))
    np.testing.assert_array_equal(np.isnan(x), np.isnan(y))
    if mask != "no common id":
        assert np.nanmax(np.abs(x - y)) <= 2**-6 * np.nanmax(np.abs(y))
    a, c = (l.cpu().numpy() for l in (l1, l2))
    seen = np.isfinite(c)
    np.testing.assert_array_equal(np.isfinite(a), seen)
    assert np.abs(a[seen] - c[seen]).max(initial=0.0) <= 2**-6
