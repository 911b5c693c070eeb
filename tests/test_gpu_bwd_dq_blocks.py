"""The query-owning kernel over dS blocks in its three sizes (128 queries and a ring of four stages below two 256-query items
per CU, 128 and three at head dimension 64 with items alike, 256 and three otherwise) at the edges of blocks, tiles and the ring, against torch autograd in fp64 on the CPU."""
import pytest

from test_gpu_parity_bwd import check, grad_errors, torch_grads_f64

pytestmark = pytest.mark.gpu

CASES = [
    # B, H, Hk, S, D, dtype, causal, wl, bshd
    (1, 2, 2, 1, 64, 0, True, -1, False),            # one query
    (1, 2, 1, 64, 128, 0, False, -1, True),          # one tile: the ring never fills
    (1, 2, 2, 129, 128, 1, True, -1, False),         # a second block of one query; three tiles
    (1, 3, 3, 191, 64, 0, True, -1, True),           # as many tiles as are requested ahead
    (1, 2, 2, 257, 64, 0, False, -1, False),         # five tiles: the ring wraps
    (1, 4, 2, 384, 128, 0, True, 70, False),         # a window: tiles outside a wave's range in the middle of a ring
    (2, 130, 130, 510, 64, 0, True, -1, False),      # 520 items: 256-query blocks, ragged
    (2, 129, 43, 512, 128, 1, False, -1, True),      # 516 items, grouped heads
    (1, 255, 255, 511, 64, 0, True, -1, False),      # 510 items: 128-query blocks, as a snake over the CUs
    (2, 256, 256, 128, 64, 1, False, -1, True),      # items alike: one 128-query block, as many tiles as requested ahead
    (1, 512, 256, 129, 64, 0, False, -1, False),     # a second block of one query, three tiles, grouped heads
    (1, 171, 171, 600, 64, 0, True, 70, True),       # a window: tiles outside a wave's range
]


@pytest.mark.parametrize("B,H,Hk,S,D,dtype,causal,wl,bshd", CASES)
def test_dq_from_blocks(fa, B, H, Hk, S, D, dtype, causal, wl, bshd):
    import torch
    g = torch.Generator(device="cuda").manual_seed(300 + S)
    dt = torch.bfloat16 if dtype else torch.float16

    def tensor(h):
        t = torch.randn((B, S, h, D) if bshd else (B, h, S, D), device="cuda", generator=g).to(dt)
        return t.transpose(1, 2) if bshd else t
    q, k, v, do = tensor(H), tensor(Hk), tensor(Hk), tensor(H)
    kw = dict(causal=causal, window_left=wl)
    o, lse = fa.flash_attention_forward(q, k, v, exact_first_rows=True, **kw)
    got = fa.flash_attention_backward(q, k, v, o, lse, do, five_products=True, poison_workspace=True, **kw)
    again = fa.flash_attention_backward(q, k, v, o, lse, do, five_products=True, poison_workspace=True, **kw)
    torch.cuda.synchronize()
    # (every K/V head is a problem of its own: the first two and the last)
    group = H // Hk
    for hk in sorted({0, min(1, Hk - 1), Hk - 1}):
        heads = slice(hk * group, (hk + 1) * group)
        want = torch_grads_f64(q[:, heads], k[:, hk:hk + 1], v[:, hk:hk + 1], do[:, heads], causal, wl, -1)
        for name, x, w in zip(("dQ", "dK", "dV"), (got[0][:, heads], got[1][:, hk:hk + 1], got[2][:, hk:hk + 1]), want):
            err = grad_errors(x.float().cpu().numpy(), w)
            print((B, H, Hk, S, D), dtype, causal, wl, bshd, hk, name, err, flush=True)
            check(err, dtype, name)
    same = all(torch.equal(a.contiguous().view(torch.int16), b.contiguous().view(torch.int16)) for a, b in zip(got, again))
    assert same
