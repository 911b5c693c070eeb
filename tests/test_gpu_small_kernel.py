"""The kernel of 32-row blocks whose waves share the keys, against the tile kernels: the same heads once as a small problem and
once among enough others that the tile kernels take the call.  Edges of its tiles (64 keys, 32 at head dimension 128), of its blocks
and of what a wave gets; every mask, with four waves and with eight; and both sides of the
rule's line (on the host: tests/test_launch_rules.py)."""
import pytest

from parity_util import small_waves


def _inputs(torch, seed, heads, kv_heads, S, Sk, D, bshd, dtype):
    g = torch.Generator(device="cuda").manual_seed(seed)
    t = [torch.randn((1, n, h, D) if bshd else (1, h, n, D), device="cuda", generator=g).to(getattr(torch, dtype))
         for h, n in ((heads, S), (kv_heads, Sk), (kv_heads, Sk))]
    return [x.transpose(1, 2) for x in t] if bshd else t


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("S,Sk,D,group,bshd,kw", [
    (33, 33, 64, 1, False, {}), (64, 64, 128, 1, False, dict(causal=True)), (65, 65, 64, 2, True, dict(causal=True)), (100, 100, 128, 1, True, {}),
    (256, 256, 64, 1, False, {}), (257, 257, 128, 4, True, dict(causal=True)), (300, 300, 64, 1, True, dict(causal=True, window_left=40)),
    (300, 300, 128, 1, False, dict(window_left=33, window_right=7)), (500, 500, 64, 1, False, dict(causal=True, window_left=0)),
    (40, 700, 64, 1, False, dict(causal=True)), (50, 75, 128, 2, True, dict(causal=True)), (96, 1111, 128, 1, False, dict(causal=True)),
    (90, 40, 64, 1, False, dict(causal=True)), (70, 200, 128, 1, True, dict(window_left=10, window_right=3)), (1700, 1700, 64, 1, False, {}),
    (130, 1900, 128, 1, True, {}), (200, 200, 64, 2, False, "slopes"), (150, 260, 128, 1, True, "slopes"),
    (70, 1600, 64, 1, False, "slopes"), (100, 900, 128, 2, True, "slopes"), (200, 3000, 64, 1, True, dict(causal=True, window_left=1700)),
    (90, 2000, 128, 1, False, dict(window_left=500, window_right=400)), (128, 128, 64, 1, False, dict(softmax_scale=1.5, causal=True)),
    (200, 200, 128, 1, False, dict(causal=True, exact_first_rows=True))])
def test_small_against_tile_kernels(fa, dtype, S, Sk, D, group, bshd, kw):
    import torch
    kv = 4 // group
    # (causal walks of 2048 queries aside, 512 blocks are the most; the other heads repeat the first four)
    times = 1 + 512 // (4 * ((S + 31) // 32))
    q, k, v = _inputs(torch, S + Sk, 4, kv, S, Sk, D, bshd, dtype)
    many = [x.repeat(times, 1, 1, 1) if not bshd else x.transpose(1, 2).repeat(times, 1, 1, 1).transpose(1, 2) for x in (q, k, v)]
    if kw == "slopes":
        kw = dict(alibi_slopes=torch.tensor([0.5, -0.25, 0.1, 0.0], device="cuda"), causal=True)
    assert small_waves(fa, q, k, **kw) > 0 and small_waves(fa, many[0], many[1], **kw) == 0
    out = torch.full_like(q, float("nan"))
    lse = torch.full((1, 4, S), float("nan"), device="cuda")
    fa.flash_attention_forward(q, k, v, out=out, lse=lse, **kw)
    o2, lse2 = fa.flash_attention_forward(*many, **kw)
    assert out.isfinite().all() and not lse.isnan().any()
    # P and O are rounded to the storage type once each, from sums in another order: a place of the larger values
    a, b = out[0].float(), o2[0].float()
    tol = 2.0 ** -9 if dtype == "float16" else 2.0 ** -6
    assert float((a - b).abs().max()) <= tol * max(1.0, float(b.abs().max())) and float((a - b).norm()) <= tol * float(b.norm())
    assert torch.equal(lse[0].isinf(), lse2[0].isinf())
    assert float((lse[0] - lse2[0]).nan_to_num(0.0, 0.0, 0.0).abs().max()) <= 1e-4 * max(1.0, float(lse2[0].nan_to_num(0.0, 0.0, 0.0).abs().max()))


@pytest.mark.gpu
@pytest.mark.parametrize("H,S,D,parts,kw", [(16, 1024, 64, 0, dict()), (51, 320, 128, 0, dict()), (8, 4096, 64, 4, dict(causal=True)), (16, 2048, 128, 4, dict(causal=True)),
                                            (53, 256, 64, 4, dict(causal=True)), (42, 256, 128, 4, dict(causal=True))])
def test_both_sides_of_the_line(fa, H, S, D, parts, kw):
    """The most heads that the small kernel takes, and one more, with which the tile kernels do: the same heads agree."""
    import ctypes
    import torch
    q, k, v = _inputs(torch, H + S, H + 1, H + 1, S, S, D, False, "float16")
    p = fa.make_params(1, H, S, D, 0x1000, 0x2000, 0x3000, 0x4000, **kw)
    got = ctypes.c_int(-1)
    assert fa.lib().fa_sched_small(ctypes.byref(p), 256, ctypes.byref(got)) == 4 and got.value == parts and small_waves(fa, q, k, **kw) == 0
    o, lse = fa.flash_attention_forward(q[:, :H], k[:, :H], v[:, :H], **kw)
    o2, lse2 = fa.flash_attention_forward(q, k, v, **kw)
    a, b = o.float(), o2[:, :H].float()
    # (as above)
    assert float((a - b).abs().max()) <= 2.0 ** -9 * max(1.0, float(b.abs().max())) and float((a - b).norm()) <= 2.0 ** -9 * float(b.norm())
    assert float((lse - lse2[:, :H]).abs().max()) <= 1e-4 * max(1.0, float(lse2.abs().max()))
    if parts:                     # (the first rows are the verifier's arithmetic in both)
        assert torch.equal(o[:, :, :32], o2[:, :H, :32]) and torch.equal(lse[:, :, :32], lse2[:, :H, :32])


@pytest.mark.gpu
def test_values_that_are_not_finite(fa):
    """An infinity or a NaN in V reaches the rows that see its key, and none in front of its 64-key tile (masked pairs of the tile
    are products with zero); in K the rows that see it become NaN, and no other."""
    import torch
    q, k, v = _inputs(torch, 5, 4, 4, 300, 300, 64, False, "float16")
    v[0, 1, 200, 3] = float("inf")
    v[0, 2, 130, 5] = float("nan")
    k[0, 3, 250] = float("nan")
    o = fa.flash_attention_forward(q, k, v, causal=True, exact_first_rows=True, return_lse=False)[0].float()
    assert o[0].isfinite().all()
    assert o[1, :192].isfinite().all() and (o[1, 200:, 3] == float("inf")).all() and o[1, 200:, :3].isfinite().all()
    assert o[2, :128].isfinite().all() and o[2, 130:, 5].isnan().all() and o[2, 130:, 6:].isfinite().all()
    assert o[3, :250].isfinite().all() and o[3, 250:].isnan().all()


@pytest.mark.gpu
@pytest.mark.parametrize("S", [256, 300])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("bshd", [False, True])
def test_logsumexp_of_rows_that_are_not_finite(fa, S, D, bshd):
    """A NaN in a key or a query: the logsumexp of the rows that see it is NaN, as their O is -- -inf says that a row saw no key -- and the
    other rows keep their bits.  A row all of whose scores are -inf has seen keys: NaN where the lengths are the regular kernels' (0 / 0,
    as they have it), while the general ones give 0."""
    import torch
    q, k, v = _inputs(torch, S + D, 4, 4, S, S, D, bshd, "float16")
    clean, clean_lse = fa.flash_attention_forward(q, k, v, causal=True, exact_first_rows=True)
    k2, q2 = k.clone(memory_format=torch.preserve_format), q.clone(memory_format=torch.preserve_format)
    k2[0, 1, 200, 3] = float("nan")
    q2[0, 2, 100, 5] = float("nan")
    for want_lse in (True, False):
        r = fa.flash_attention_forward(q2, k2, v, causal=True, exact_first_rows=True, return_lse=want_lse)
        o, lse = r if want_lse else (r, None)
        nan = torch.zeros((1, 4, S), dtype=torch.bool, device="cuda")
        nan[0, 1, 200:] = True
        nan[0, 2, 100] = True
        assert bool(o[nan].isnan().all()) and torch.equal(o[~nan], clean[~nan])
        if want_lse:
            assert bool(lse[nan].isnan().all()) and torch.equal(lse[~nan], clean_lse[~nan])
    q.abs_().clamp_(min=0.1)
    k[0, 1] = float("-inf")
    o, lse = fa.flash_attention_forward(q, k, v, causal=True, exact_first_rows=True)
    assert bool((lse[0, 1] == float("-inf")).all()) and bool(o[0, [0, 2, 3]].isfinite().all())
    assert bool(o[0, 1].isnan().all() if S % 128 == 0 else (o[0, 1] == 0).all())


@pytest.mark.gpu
def test_sharp_scores(fa):
    """Scores of a standard deviation of 16: reference points far apart between the waves of a block."""
    import torch
    for D in (64, 128):
        q, k, v = _inputs(torch, 6, 4, 4, 400, 400, D, False, "float16")
        q = q * 16
        o = fa.flash_attention_forward(q, k, v, return_lse=False).double()
        p = torch.softmax((q.double() @ k.double().transpose(-1, -2)) / D ** 0.5, dim=-1)
        ref = p @ v.double()
        assert float((o - ref).norm() / ref.norm()) <= 5e-4
