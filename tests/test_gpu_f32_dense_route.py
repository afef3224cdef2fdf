"""fp32 forward through dense Q, K and V: which calls ask for the room (no GPU needed), and that the route agrees with the kernels that
rebuild every tile from the factors, over masks, strides, and row counts around their blocks.

Both are held to the 1e-4 / 1e-5 (logsumexp) of the fp32 kernels against the oracle; they differ in the order of the sums over the
ranks alone, and agree to the same."""

import ctypes

import numpy as np
import pytest
import torch

from conftest import segment_ids
from test_abi import _forward_call


@pytest.mark.parametrize(
    "B,H,D,lq,lk,rk,dense",
    [
        (1, 8, 64, 300, 300, 1, False),
        (2, 16, 128, 699, 699, 2, False),
        (2, 16, 128, 700, 700, 2, True),
        (2, 16, 128, 700, 3501, 2, False),
        (1, 8, 64, 1499, 1499, 2, False),
        (1, 8, 64, 1500, 1500, 2, True),
        (3, 43, 128, 1500, 1500, 2, False),  # 129 (batch, head) pairs, and no multiple of eight heads
        (2, 72, 128, 1500, 1500, 2, False),
        (1, 8, 128, 16, 300, 3, False),
        (1, 8, 128, 17, 300, 3, True),
        (5, 16, 128, 32, 300, 8, False),
        (5, 16, 128, 33, 300, 8, True),
        (5, 16, 64, 256, 300, 4, False),
        (5, 16, 64, 257, 300, 4, True),
        (1, 8, 64, 40, 699, 4, False),
        (1, 8, 64, 40, 700, 4, True),
        (1, 5, 64, 400, 700, 8, False),      # heads in no groups of eight
        (1, 32, 128, 64, 131071, 4, True),   # the last dense entry below 2 GiB, which the kernel of 32 rows can address
        (1, 32, 128, 64, 131072, 4, False),
        (1, 32, 128, 64, 140000, 4, False),
        (2, 64, 64, 17, 131072, 8, False),
        (9, 32, 128, 64, 140000, 4, True),   # 576 workgroups of 32 rows: on the factors 256 rows too
    ],
)
def test_which_calls_ask_for_it(B, H, D, lq, lk, rk, dense):
    from tpa import _dispatch as d

    lib = d.load_library()
    fake = d.TpaFactor(256, 8, 8, 8)
    call = _forward_call(B=B, H=H, D=D, lq=lq, lk=lk, rk=rk, dtype=d.TPA_DTYPE_F32, qa=fake, qb=fake, ka=fake, kb=fake, va=fake, vb=fake)
    if lq <= 16:
        call.kernel = d.KERNEL_MFMA
        call.q_segment_ids = call.kv_segment_ids = 256  # not a decode
    need = lib.tpa_fwd_call_workspace_bytes(ctypes.byref(call))
    slot = lambda n: (n + 63) // 64 * 256
    assert need == (slot(B * lq * H * D) + 2 * slot(B * lk * H * D) if dense else 0)
    assert need <= lib.tpa_fwd_best_workspace_bytes(B, lq, lk, H, D, D, 6, rk)


@pytest.mark.parametrize(
    "B,H,D,lq,lk,rq,rk,call,dense",
    [
        (4, 16, 128, 100, 100, 6, 3, dict(causal=1), False),    # 32 rows: one step of four waves
        (4, 16, 128, 100, 100, 6, 8, dict(causal=1), True),
        (2, 16, 128, 200, 200, 6, 4, dict(causal=1), True),     # two
        (12, 32, 128, 40, 40, 2, 3, dict(causal=1), False),     # 256 rows, Q of two ranks
        (12, 32, 128, 40, 40, 16, 3, dict(causal=1), True),
        (2, 64, 64, 307, 307, 2, 4, dict(), False),
        (2, 64, 64, 307, 307, 16, 4, dict(), True),
        (4, 32, 128, 135, 135, 2, 3, dict(), False),            # 128 rows
        (4, 32, 128, 135, 135, 16, 3, dict(), True),
        (4, 32, 128, 256, 1000, 2, 3, dict(causal=2), True),
        (4, 32, 128, 256, 1000, 2, 3, dict(causal=1), False),   # a quarter of the keys in reach
        (4, 16, 128, 40, 1500, 6, 3, dict(causal=1), False),    # the same of 32 rows
        (4, 16, 128, 40, 1500, 6, 3, dict(causal=1, causal_offset=1460), True),
        (4, 16, 128, 40, 1500, 6, 3, dict(causal=1, causal_offset=-40), False),
        (45, 40, 128, 100, 317, 4, 3, dict(q_segment_ids=256, kv_segment_ids=256), False),  # documents: 228 of 317 keys
        (1, 8, 128, 65537, 65537, 6, 3, dict(causal=1), True),  # more blocks than are looked at
    ],
)
def test_calls_that_would_not_win_by_it(B, H, D, lq, lk, rq, rk, call, dense):
    from tpa import _dispatch as d

    lib = d.load_library()
    fake = d.TpaFactor(256, 8, 8, 8)
    call = _forward_call(B=B, H=H, D=D, lq=lq, lk=lk, rq=rq, rk=rk, dtype=d.TPA_DTYPE_F32, qa=fake, qb=fake, ka=fake, kb=fake, va=fake, vb=fake, **call)
    slot = lambda n: (n + 63) // 64 * 256
    assert lib.tpa_fwd_call_workspace_bytes(ctypes.byref(call)) == (slot(B * lq * H * D) + 2 * slot(B * lk * H * D) if dense else 0)


@pytest.mark.parametrize("name", ["qa", "qb", "ka", "kb", "va", "vb"])
def test_rows_that_the_launch_refuses_ask_for_nothing(name):
    """Rows of factors that start between 16 bytes, and more batch entries than the launch has room for: such a call runs on the factors."""
    from tpa import _dispatch as d

    lib = d.load_library()
    fake = d.TpaFactor(256, 8, 8, 8)
    factors = dict(qa=fake, qb=fake, ka=fake, kb=fake, va=fake, vb=fake)
    make = lambda B=1, **f: _forward_call(B=B, H=8, D=128, lq=300, lk=3000, rk=8, dtype=d.TPA_DTYPE_F32, **{**factors, **f})
    room = lambda call: lib.tpa_fwd_call_workspace_bytes(ctypes.byref(call))
    assert room(make()) > 0
    assert room(make(**{name: d.TpaFactor(256, 8, 9, 8)})) == 0
    assert room(make(**{name: d.TpaFactor(260, 8, 8, 8)})) == 0
    assert room(make(B=65536)) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["concatenated", "split", "ranks first"])
@pytest.mark.parametrize("mask", ["none", "causal", "offset", "bottom right", "lengths", "packed", "ids in no order", "no common id"])
@pytest.mark.parametrize("b,h,d,lq,lk,rk", [(1, 8, 64, 40, 705, 4), (2, 40, 64, 257, 300, 3), (3, 8, 128, 33, 100, 8), (2, 16, 128, 700, 720, 2), (1, 16, 128, 129, 400, 5)])
def test_both_routes_agree(gpu, b, h, d, lq, lk, rk, mask, layout):
    from tpa import tpa

    gen = torch.Generator(device="cpu").manual_seed(lq)

    def factors(l, r):
        x = (torch.randn((b, l, r, h + d), generator=gen) / r**0.5).to(gpu)
        parts = x[..., :h], x[..., h:]
        if layout == "split":
            return tuple(p.contiguous() for p in parts)
        if layout == "ranks first":
            return tuple(p.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3) for p in parts)
        return parts

    args = list(factors(lq, 6) + factors(lk, rk) + factors(lk, rk))
    kw = dict(sm_scale=d**-0.5, causal=mask in ("causal", "offset", "packed"), kernel=2)
    if mask == "offset":
        kw["causal_offset"] = lk - lq
    if mask == "bottom right":
        kw["causal"] = tpa.CAUSAL_BOTTOM_RIGHT
    if mask in ("lengths", "bottom right"):
        lengths = [lk - 77 * i for i in range(b)]
        kw["kv_lengths"] = torch.tensor(lengths, dtype=torch.int32, device=gpu)
        for n in range(2, 6):  # padding is never met
            args[n] = args[n].clone(memory_format=torch.preserve_format)
            for i, x in enumerate(lengths):
                args[n][i, x:] = float("nan")
    if mask == "packed":
        ids = torch.from_numpy(segment_ids(max(lq, lk), 97, b)).to(gpu)
        kw["q_segment_ids"], kw["kv_segment_ids"] = ids[:, :lq].contiguous(), ids[:, :lk].contiguous()
    if mask in ("ids in no order", "no common id"):
        kw["q_segment_ids"] = torch.randint(0, 3, (b, lq), generator=gen, dtype=torch.int32).to(gpu)
        kw["kv_segment_ids"] = torch.randint(0, 3, (b, lk), generator=gen, dtype=torch.int32).to(gpu) + (5 if mask == "no common id" else 0)
    (o1, l1), (o2, l2) = (tpa.tpa_factors(*args, use_workspace=w, **kw) for w in (True, False))
    x, y = (o.cpu().numpy().astype(np.float64) for o in (o1, o2))
    np.testing.assert_array_equal(np.isnan(x), np.isnan(y))
    if mask != "no common id":
        assert np.nanmax(np.abs(x - y)) <= 1e-4
    a, c = (l.cpu().numpy() for l in (l1, l2))
    seen = np.isfinite(c)
    np.testing.assert_array_equal(np.isfinite(a), seen)
    assert np.abs(a[seen] - c[seen]).max(initial=0.0) <= 1e-5


@pytest.mark.gpu
def test_values_that_do_not_split(gpu):
    """Infinities, NaN and magnitudes at both ends of fp32 in K and V: the second walk meets them on the dense arrays too."""
    from tpa import tpa

    gen = torch.Generator(device="cpu").manual_seed(3)
    b, h, d, l, rk = 1, 8, 128, 300, 4
    make = lambda r, x: (torch.randn((b, l, r, x), generator=gen) / r**0.5).to(gpu)
    args = [make(6, h), make(6, d), make(rk, h), make(rk, d), make(rk, h), make(rk, d)]
    for at, value in ((10, float("inf")), (70, 1e-38), (130, 3e38), (200, float("nan"))):
        args[5][0, at, 0, 5] = value
    args[3][0, 250] *= 1e-36
    kw = dict(sm_scale=d**-0.5, kernel=2, causal=True)
    (o1, l1), (o2, l2) = (tpa.tpa_factors(*args, use_workspace=w, **kw) for w in (True, False))
    torch.testing.assert_close(o1, o2, rtol=1e-4, atol=1e-4, equal_nan=True)
    torch.testing.assert_close(l1, l2, rtol=0, atol=1e-5)
