"""The dense arrays of a forward call hold no more keys than its lengths and its mask let a query see: whatever a workspace of the test's own
was filled with, and whatever lies in the padding of the cache, the results are the same bits."""

import ctypes

import pytest
import torch


@pytest.mark.gpu
@pytest.mark.parametrize("mask", ["lengths", "bottom right", "short offset", "before the keys", "packed"])
@pytest.mark.parametrize(
    "dtype,b,h,d,lq,lk,rk",
    [
        (torch.bfloat16, 5, 8, 64, 300, 700, 4),
        (torch.bfloat16, 5, 16, 128, 40, 1100, 8),
        (torch.bfloat16, 1, 8, 64, 33, 4000, 4),  # the keys in ranges
        (torch.bfloat16, 2, 8, 128, 600, 900, 2),
        (torch.float32, 5, 8, 64, 90, 705, 16),
        (torch.float32, 3, 16, 128, 140, 400, 8),
    ],
)
def test_whatever_fills_the_workspace(gpu, dtype, b, h, d, lq, lk, rk, mask):
    from tpa import _dispatch as d_
    from tpa import tpa

    gen = torch.Generator(device="cpu").manual_seed(lk)
    make = lambda l, r, x: (torch.randn((b, l, r, x), generator=gen) / r**0.5).to(gpu, dtype)
    args = [make(l, r, x) for l, r in ((lq, 6), (lk, rk), (lk, rk)) for x in (h, d)]
    kw = dict(sm_scale=d**-0.5, kernel=2, causal=mask in ("short offset", "before the keys"))
    ends = [lk] * b
    if mask == "short offset":
        kw["causal_offset"] = 77
        ends = [min(lk, lq + 77)] * b
    if mask == "before the keys":
        kw["causal_offset"] = -lq // 2
        ends = [min(lk, lq - -(-lq // 2))] * b
    if mask in ("lengths", "bottom right", "packed"):
        ends = [lk - 130, 1, 64, 65, 0][:b]
        kw["kv_lengths"] = torch.tensor(ends, dtype=torch.int32, device=gpu)
    if mask == "bottom right":
        kw["causal"] = tpa.CAUSAL_BOTTOM_RIGHT
    if mask == "packed":
        ids = (torch.arange(lk, dtype=torch.int32)[None] // 97).expand(b, lk).contiguous().to(gpu)
        kw["q_segment_ids"], kw["kv_segment_ids"] = ids[:, :lq].contiguous(), ids

    # the library is called with a workspace of our own: what lies in it is certain, and that the call uses it
    lib = d_.load_library()
    ids = [kw.get(n) for n in ("q_segment_ids", "kv_segment_ids", "kv_lengths")]
    pointer = lambda t: None if t is None else t.data_ptr()

    def run(filling, byte):
        xs = list(args)
        for n in range(2, 6):
            xs[n] = xs[n].clone()
            for i, x in enumerate(ends):
                xs[n][i, x:] = filling
        o = torch.zeros((b, lq, h, d), dtype=dtype, device=gpu)
        lse = torch.zeros((b, h, lq), dtype=torch.float32, device=gpu)
        call = d_.TpaFwdArgs(**{n: d_.factor(x) for n, x in zip(("qa", "qb", "ka", "kb", "va", "vb"), xs)},
                             q_segment_ids=pointer(ids[0]), kv_segment_ids=pointer(ids[1]), kv_lengths=pointer(ids[2]), o=o.data_ptr(), lse=lse.data_ptr(),
                             B=b, lq=lq, lk=lk, H=h, dk=d, dv=d, rq=6, rk=rk, dtype=d_.dtype_code(dtype), sm_scale=kw["sm_scale"],
                             causal=int(kw["causal"]), causal_offset=kw.get("causal_offset", 0), kernel=kw["kernel"])
        need = lib.tpa_fwd_call_workspace_bytes(ctypes.byref(call))
        dense = b * h * d * (lq + 2 * lk) * o.element_size()
        assert need >= dense
        room = torch.full((need + 256,), byte, dtype=torch.uint8, device=gpu)
        call.workspace, call.workspace_bytes = room.data_ptr() + (-room.data_ptr()) % 256, need
        assert lib.tpa_fwd(ctypes.byref(call), d_.current_stream_ptr(gpu)) == 0
        assert not (room[: dense // 2] == byte).all()
        return o, lse

    (o1, l1), (o2, l2) = run(0.0, 0), run(float("nan"), 255)  # bytes of ones are NaN in either type
    assert torch.equal(l1, l2)
    assert torch.equal(o1.nan_to_num(nan=1e9), o2.nan_to_num(nan=1e9))
