"""The pass that makes delta and the rescaled logsumexp for the five-product backward (64 rows of a head per workgroup at head
dimension 128, 128 at 64; the rows of all heads one behind the other where a head has at most a quarter of that) at the edges of
those pieces, in both orders of its workgroups and beyond the 65536 of a launch, against torch autograd in fp64 on the CPU."""
import pytest

import test_gpu_bwd_dq_blocks as blocks

pytestmark = pytest.mark.gpu

CASES = [
    # B, H, Hk, S, D, dtype, causal, wl, bshd
    (2, 3, 3, 63, 128, 0, True, -1, False),          # a piece, a row short
    (3, 4, 2, 65, 128, 1, True, -1, True),           # a second piece of one row, heads inside rows, several batches
    (3, 5, 5, 127, 64, 0, False, -1, True),
    (2, 3, 1, 129, 64, 1, True, -1, False),
    (2, 3, 3, 128, 64, 0, True, -1, True),           # whole pieces
    (40, 1640, 1640, 1, 64, 0, True, -1, True),      # 65600 heads of one row
    (40, 1640, 1640, 65, 64, 0, True, -1, True),     # 65600 workgroups' work
    # short sequences, rows of all heads one behind the other: up to 32 rows at head dimension 64, 16 at 128
    (3, 5, 5, 32, 64, 1, False, -1, True),
    (3, 5, 5, 33, 64, 0, True, -1, True),            # (the first length that is not)
    (3, 4, 2, 16, 128, 0, True, -1, True),
    (2, 3, 3, 17, 128, 1, True, -1, False),
    (7, 3, 1, 5, 128, 1, False, -1, True),           # 105 rows: a last workgroup that is not full
    (5, 13108, 13108, 16, 128, 0, True, -1, False),  # 1048640 rows, 16 to a workgroup: beyond a launch's 65536
]


@pytest.mark.parametrize("B,H,Hk,S,D,dtype,causal,wl,bshd", CASES)
def test_prepare(fa, B, H, Hk, S, D, dtype, causal, wl, bshd):
    blocks.test_dq_from_blocks(fa, B, H, Hk, S, D, dtype, causal, wl, bshd)
