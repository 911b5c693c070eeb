"""The key-owning kernel of the five-product form at head dimension 64, whose workgroups own 128 keys (two to a compute
unit), at the edges of those blocks and of a launch that fills the chip once, against torch autograd in fp64 on the CPU."""
import pytest

import test_gpu_bwd_dq_blocks as blocks

pytestmark = pytest.mark.gpu

CASES = [
    # B, H, Hk, S, D, dtype, causal, wl, bshd
    (1, 9, 9, 127, 64, 0, True, -1, False),          # one block, a key short
    (1, 9, 3, 129, 64, 1, False, -1, True),          # a second block of one key, grouped heads
    (2, 256, 256, 128, 64, 0, True, -1, False),      # 512 items: one round
    (1, 257, 257, 130, 64, 1, True, -1, True),       # 514 items: a snake over the resident workgroups, ragged
    (1, 200, 200, 300, 64, 0, True, 50, False),      # a window, three blocks
]


@pytest.mark.parametrize("B,H,Hk,S,D,dtype,causal,wl,bshd", CASES)
def test_key_blocks(fa, B, H, Hk, S, D, dtype, causal, wl, bshd):
    blocks.test_dq_from_blocks(fa, B, H, Hk, S, D, dtype, causal, wl, bshd)
