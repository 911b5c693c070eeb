"""The first rows of every head in workgroups of their own (launches of one workgroup per work item) give the bits that they give
behind the tile loops of the list's items (the fixed order, sched 2), wherever the rows end: one block and several, lengths
below a part, queries behind a few earlier keys, other storage orders, every option that the path has."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("H,Hk,S,S_kv,D,bshd,kw", [
    # (two batch entries; more 32-row blocks than the kernel for small problems takes)
    (140, 140, 33, 33, 64, False, {}), (140, 70, 33, 33, 128, True, {}), (100, 100, 128, 128, 64, False, {}), (100, 25, 128, 128, 128, True, {}),
    (40, 10, 256, 256, 128, True, {}), (30, 30, 300, 300, 64, False, dict(window_left=5)), (25, 25, 384, 384, 128, False, dict(window_left=40)),
    (70, 70, 100, 131, 64, False, {}), (140, 140, 40, 60, 128, True, {}),
    (8, 8, 256, 256, 64, True, dict(dropout_prob=0.3, seed=5)), (4, 4, 200, 200, 128, False, dict(dropout_prob=0.3, seed=5)),
    (4, 4, 1, 1, 64, False, dict(dropout_prob=0.3, seed=5)), (4, 2, 31, 31, 64, True, dict(dropout_prob=0.3, seed=5)), (4, 4, 9, 40, 128, True, dict(dropout_prob=0.3, seed=5)),
    (100, 50, 128, 128, 64, False, "slopes"), (50, 50, 170, 170, 128, True, "slopes"),
    (300, 300, 128, 128, 64, False, {}), (500, 500, 100, 100, 128, False, {})])             # (none apart)
def test_rows_apart_are_the_bits_of_rows_in_items(fa, dtype, H, Hk, S, S_kv, D, bshd, kw):
    import torch
    g = torch.Generator(device="cuda").manual_seed(S + H)
    q, k, v = (torch.randn((2, n, h, D) if bshd else (2, h, n, D), device="cuda", generator=g).to(getattr(torch, dtype))
               for h, n in ((H, S), (Hk, S_kv), (Hk, S_kv)))
    if bshd:
        q, k, v = (t.transpose(1, 2) for t in (q, k, v))
    if kw == "slopes":
        kw = dict(alibi_slopes=torch.linspace(-0.5, 0.5, H, device="cuda"))
    results = []
    for sched in (fa.FA_SCHED_AUTO, fa.FA_SCHED_DISPATCH, fa.FA_SCHED_PERSISTENT):
        out = torch.full_like(q, float("nan"))
        lse = torch.full((2, H, S), float("nan"), device="cuda")
        fa.flash_attention_forward(q, k, v, causal=True, out=out, lse=lse, sched=sched, **kw)
        torch.cuda.synchronize()
        assert not out.isnan().any() and not lse.isnan().any()
        results.append((out.contiguous().view(torch.int16), lse.view(torch.int32)))
    for o, l in results[:2]:
        assert torch.equal(o, results[2][0]) and torch.equal(l, results[2][1])
