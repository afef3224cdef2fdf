"""Key ranges of a decode from rank 4 on: how many there are with the room for their partials and without, at the edges of a block per
wave, and that the merge takes all of them.

Ranges are merged by exact powers of two and a range's blocks go to its waves in turn, so calls that differ in the number of ranges
differ in the order of fp32 sums alone: a result may round to the neighbouring bf16 value (2^-7 of its size, or 2^-12 of the row's
largest where terms cancel), fp32 results agree to the 1e-4 of the other fp32 tests, the logsumexp to 1e-5."""

import ctypes

import pytest
import torch


def _call(b, lq, lk, h, d, rk, bf16=True, splits=0):
    from tpa import _dispatch as disp

    fake = disp.TpaFactor(256, 8, 8 * rk, 8)
    return disp.TpaFwdArgs(qa=fake, qb=fake, ka=fake, kb=fake, va=fake, vb=fake, o=256, B=b, lq=lq, lk=lk, H=h, dk=d, dv=d, rq=6, rk=rk,
                           dtype=disp.TPA_DTYPE_BF16 if bf16 else disp.TPA_DTYPE_F32, sm_scale=1.0, num_splits=splits)


@pytest.mark.parametrize(
    "b,lq,lk,h,d,rk,bf16,ranges",
    [
        (1, 1, 700, 16, 128, 8, True, 44),    # a block of four keys per wave
        (1, 1, 704, 16, 128, 8, True, 44),
        (1, 1, 705, 16, 128, 8, True, 45),
        (1, 1, 700, 16, 128, 4, True, 22),
        (1, 1, 700, 16, 128, 2, True, 11),    # as by the sizes alone
        (1, 1, 700, 64, 64, 4, True, 22),     # one set of columns
        (1, 2, 700, 64, 64, 4, True, 22),     # two sets of columns
        (1, 1, 700, 64, 64, 8, True, 44),
        (1, 1, 700, 16, 64, 4, False, 22),
        (1, 1, 2016, 16, 64, 4, True, 63),    # as many as that pays for, in blocks of eight keys
        (1, 1, 2500, 16, 64, 4, True, 64),
        (1, 2, 8000, 32, 64, 4, True, 125),   # by the sizes alone
        (1, 1, 7724, 8, 64, 8, True, 128),
        (1, 1, 7724, 8, 64, 8, False, 256),
        (4, 1, 9000, 32, 128, 8, True, 64),   # a workgroup per compute unit
        (300, 1, 9000, 32, 128, 8, True, 1),
        (1, 1, 100000, 128, 128, 32, True, 64),
        (1, 1, 700, 16, 128, 6, True, 11),    # a rank no matrix-core kernel takes
    ],
)
def test_room_for_a_block_per_wave(b, lq, lk, h, d, rk, bf16, ranges):
    from tpa import _dispatch as disp

    lib = disp.load_library()
    need = lib.tpa_decode_call_workspace_bytes(ctypes.byref(_call(b, lq, lk, h, d, rk, bf16)))
    assert need == b * lq * h * (d + 2) * 4 * ranges
    assert need >= lib.tpa_decode_workspace_bytes(b, lq, lk, h, d, 0)
    assert lib.tpa_decode_call_workspace_bytes(ctypes.byref(_call(b, lq, lk, h, d, rk, bf16, 3))) == lib.tpa_decode_workspace_bytes(b, lq, lk, h, d, 3)
    if lq <= 16 and lk >= 1024:
        assert need <= lib.tpa_fwd_best_workspace_bytes(b, lq, lk, h, d, d, 6, rk)


@pytest.mark.gpu
@pytest.mark.parametrize("h,d,rk", [(16, 64, 4), (32, 64, 8), (8, 128, 4), (64, 64, 16), (32, 128, 32)])
@pytest.mark.parametrize("lengths", [[317, 200, 158, 250] * 7, [1519, 760], [32, 33, 64, 65, 31, 1, 0, 1000], [128 * 32], [16 * i + 1 for i in range(64)]])
def test_short_ranges_are_whole_rounds(gpu, lengths, h, d, rk):
    """Lengths of which the ranges' share lies at, below and between rounds of blocks: every entry is what it is alone."""
    from tpa import tpa

    gen = torch.Generator(device="cpu").manual_seed(len(lengths))
    b, lk, lq = len(lengths), max(lengths), 2
    make = lambda n, r, x: (torch.randn((b, n, r, x), generator=gen) / r**0.5).to(gpu, torch.bfloat16)
    args = [make(n, r, x) for n, r in ((lq, 6), (lk, rk), (lk, rk)) for x in (h, d)]
    kw = dict(sm_scale=d**-0.5, kernel=2)
    o, lse = tpa.tpa_decode(*args, kv_lengths=torch.tensor(lengths, dtype=torch.int32, device=gpu), **kw)
    for i in sorted({0, b // 2, b - 1, lengths.index(max(lengths)), lengths.index(min(lengths))}):
        if not lengths[i]:
            assert o[i].isnan().all() and lse[i].isneginf().all()
            continue
        want, want_lse = tpa.tpa_decode(*(x[i : i + 1, : (lengths[i] if n > 1 else lq)] for n, x in enumerate(args)), num_splits=1, **kw)
        got, want = o[i].float(), want[0].float()
        assert ((got - want).abs() <= 2**-7 * want.abs() + 2**-12 * want.abs().amax(-1, keepdim=True)).all()
        assert torch.allclose(lse[i], want_lse[0], atol=1e-5, rtol=0)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["plain", "lengths", "paged"])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize(
    "b,lq,lk,h,d,rk",
    [(1, 1, 704, 16, 128, 8), (2, 2, 705, 32, 128, 8), (1, 4, 321, 8, 64, 4), (3, 1, 1000, 64, 64, 16), (1, 3, 512, 16, 128, 4), (2, 1, 130, 24, 128, 32)],
)
def test_any_room_gives_one_result(gpu, b, lq, lk, h, d, rk, dt, kind):
    from tpa import tpa

    gen = torch.Generator(device="cpu").manual_seed(lk)
    make = lambda l, r, x: (torch.randn((b, l, r, x), generator=gen) / r**0.5).to(dt).to(gpu)
    q, kv = (make(lq, 6, h), make(lq, 6, d)), [make(lk, rk, x) for x in (h, d, h, d)]
    kw = dict(sm_scale=d**-0.5, kernel=2)
    capacity = lk
    if kind != "plain":
        kw["kv_lengths"] = torch.tensor([lk - 37 * i for i in range(b)], dtype=torch.int32, device=gpu)
        kw["causal"] = tpa.CAUSAL_BOTTOM_RIGHT
    else:
        kw.update(causal=True, causal_offset=lk - lq)
    if kind == "paged":
        capacity = -(-lk // 64) * 64
        kv = [torch.cat([x, torch.full_like(x[:, : capacity - lk], float("nan"))], 1).reshape(-1, 64, *x.shape[2:]).contiguous() for x in kv]
        order = torch.randperm(kv[0].shape[0], generator=gen)
        kv = [x[order.to(gpu)].contiguous() for x in kv]
        kw["page_table"] = torch.argsort(order).to(torch.int32).view(b, -1).to(gpu)
    one, lse1 = tpa.tpa_decode(*q, *kv, num_splits=1, **kw)
    told = tpa.decode_workspace_bytes(b, lq, capacity, h, d)
    for room in (None, told, 2 * told):
        ws = None if room is None else torch.full((room,), 0xFF, dtype=torch.uint8, device=gpu)
        o, lse = tpa.tpa_decode(*q, *kv, workspace=ws, **kw)
        x, y = o.double(), one.double()
        if dt == torch.bfloat16:
            assert bool(((x - y).abs() <= torch.maximum(2.0**-7 * y.abs(), 2.0**-12 * y.abs().amax(-1, keepdim=True))).all()), room
        else:
            torch.testing.assert_close(x, y, rtol=1e-4, atol=1e-4)
        torch.testing.assert_close(lse, lse1, rtol=0, atol=1e-5)
