"""fp32 matrix-core kernels of 32 rows with eight waves (head size 64, 384 and more keys or rows streamed) at the edges of
that rule, ranks past the six whose loads travel together, and more than 512 causal workgroups."""

import pytest

from test_gpu_f32_blocks import test_f32_workgroup_sizes as check_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(
    "b,lq,lk,h,d,rq,rk,causal,seg",
    [
        (1, 383, 384, 2, 64, 7, 1, True, None),    # eight waves forward and for dQ, four for dK and dV
        (2, 385, 383, 1, 64, 6, 3, False, None),   # the other way round; a block of one row
        (1, 400, 420, 2, 64, 13, 2, True, 90),     # windows: most waves have no tile
        (1, 420, 420, 2, 64, 2, 4, False, 200),
        (3, 770, 770, 8, 64, 6, 2, True, None),    # 600 workgroups of 32 rows
        (1, 390, 390, 2, 128, 7, 2, True, None),   # head size 128 keeps four
    ],
)
def test_eight_waves(gpu, b, lq, lk, h, d, rq, rk, causal, seg):
    check_problem(gpu, b, lq, lk, h, d, rq, rk, causal, seg)
