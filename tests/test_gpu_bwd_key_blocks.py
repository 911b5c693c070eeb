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


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("B,H,Hk,S,bshd", [(1, 130, 130, 512, False), (2, 72, 36, 1024, True), (3, 100, 100, 256, False)])
def test_dropout_items_of_the_seven_products_as_a_snake(fa, dtype, B, H, Hk, S, bshd):
    """128-wide, causal, dropout, seven products: between one and sixteen items per compute unit the workgroups walk several
    items each (260 and 288 of the key-owning kernel; 300 of one length), against the five products, which have kernels of
    their own.  Both round P and dS to the storage type, u = 2^-11 or 2^-8, at other places: at most 2 u between them in the
    2-norm."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(S + H)
    dt = torch.float16 if dtype == "fp16" else torch.bfloat16
    q, k, v, do = (torch.randn((B, n, S, 128), generator=g, device="cuda").to(dt) for n in (H, Hk, Hk, H))
    if bshd:
        q, k, v, do = (x.transpose(1, 2).contiguous().transpose(1, 2) for x in (q, k, v, do))
    kw = dict(causal=True, dropout_prob=0.2, seed=11)
    o, lse = fa.flash_attention_forward(q, k, v, exact_first_rows=True, **kw)
    seven = fa.flash_attention_backward(q, k, v, o, lse, do, five_products=False, poison_workspace=True, **kw)
    five = fa.flash_attention_backward(q, k, v, o, lse, do, five_products=True, **kw)
    again = fa.flash_attention_backward(q, k, v, o, lse, do, five_products=False, **kw)
    torch.cuda.synchronize()
    u = 2.0 ** -11 if dtype == "fp16" else 2.0 ** -8
    for a, b, c in zip(seven, five, again):
        assert torch.equal(a, c)
        assert float((a.double() - b.double()).norm() / b.double().norm()) <= 2 * u
