"""How many key ranges a decode has and how much workspace callers are told, without a GPU."""

import pytest

SCRATCH = 8 << 20  # of tpa_decode_noalloc


def _lib():
    from tpa import _dispatch

    return _dispatch.load_library()


@pytest.mark.parametrize("b,lq,lk,want", [(1, 4, 32768, 256), (1, 3, 32768, 256), (1, 8, 32768, 128), (6, 4, 32768, 43), (1, 2, 32768, 256), (64, 4, 8192, 4)])
def test_eight_heads_fill_the_chip_with_four_rows_to_a_workgroup(b, lq, lk, want):
    """8 heads of four query rows lie side by side in one workgroup's columns: the ranges make 256 workgroups of them."""
    assert _lib().tpa_decode_default_splits(b, lq, lk, 8) == want


def test_the_fixed_array_holds_what_it_held():
    """Counting four rows to a workgroup adds ranges, but none beyond what the scratch memory of tpa_decode_noalloc holds where two
    rows to a workgroup fitted."""
    lib = _lib()
    for lq in (3, 4, 5, 7, 8, 12, 16, 33, 63, 64):
        for b in (1, 2, 3, 7, 15, 16, 31, 63, 64, 85, 127, 200, 255, 256):
            for lk in (64, 1000, 8192, 100000):
                groups = b * ((lq + 1) // 2)
                want = -(-256 // groups)
                room = SCRATCH // (b * lq * 8 * 130 * 4)
                two = 1 if groups >= 256 else max(1, min(want, -(-lk // 256)), min(want, -(-lk // 64), room))
                now = lib.tpa_decode_default_splits(b, lq, lk, 8)
                assert now >= two, (b, lq, lk)
                need = lib.tpa_decode_workspace_bytes(b, lq, lk, 8, 128, 0)
                assert need == b * lq * now * 8 * 130 * 4
                assert need <= SCRATCH or now == two, (b, lq, lk)


@pytest.mark.parametrize("h", [1, 4, 7, 16, 24, 32, 64])
def test_other_head_counts_have_two_rows_to_a_workgroup(h):
    lib = _lib()
    for b, lq in ((1, 1), (1, 4), (3, 8), (20, 5)):
        groups = b * ((lq + 1) // 2) * -(-h // 32)
        want = -(-256 // groups)
        room = SCRATCH // (b * lq * h * 130 * 4)
        assert lib.tpa_decode_default_splits(b, lq, 5000, h) == max(1, min(want, -(-5000 // 256)), min(want, -(-5000 // 64), room))
