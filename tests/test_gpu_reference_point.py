"""The reference point of the forward kernels' exponentials where it has to move inside the tile loop: scores that grow
along the keys by far more than one tile's sum may hold, rows whose first visible keys lie in their second tile, and NaN.

Against the same attention in 64 bits.  Tolerances: P and O are rounded to the storage type once each, u = 2^-11 (fp16) or
2^-8 (bf16) at most per value.  With growing scores a few keys carry a row, so O is as far off as two roundings of its
largest terms: 4 u of the row's largest |V| for single values, 1.5 u in the 2-norm (about u expected)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    # B, H, Hk, S, D, dtype, causal, wl, bshd, growth per key (in units of the scaled score); the kernels named are those that run the
    # case, or copies of it where it is small
    (1, 2, 2, 512, 64, "fp16", True, -1, False, 0.4),      # every tile moves the reference point
    (1, 2, 2, 512, 128, "bf16", False, -1, False, 0.4),
    (1, 2, 1, 512, 128, "fp16", True, -1, True, 0.15),     # some do; strided kernels
    (1, 2, 2, 500, 64, "bf16", True, -1, False, 0.3),      # general kernels
    (1, 2, 2, 500, 128, "fp16", False, -1, True, 0.3),
    (2, 16, 16, 2048, 128, "fp16", True, -1, False, 0.2),  # eight-wave workgroups
    (2, 64, 64, 1200, 64, "fp16", True, 96, False, 0.2),   # windows: the first keys of a row in its block's second tile
    (1, 2, 2, 1024, 128, "fp16", True, 65, False, 0.1),
    (1, 2, 2, 512, 64, "fp16", False, -1, False, -0.4),    # the first tile holds the maximum: nothing moves
]


def _inputs(B, H, Hk, S, D, dtype, growth, bshd, seed):
    import torch
    g = torch.Generator().manual_seed(seed)
    dt = torch.bfloat16 if dtype == "bf16" else torch.float16
    q, k, v = (torch.randn((B, n, S, D), generator=g) for n in (H, Hk, Hk))
    q[..., 0] = 8.0
    k[..., 0] = torch.arange(S) * (growth * D ** 0.5 / 8.0)          # score of key j: growth * j + noise
    q, k, v = (x.to(dt) for x in (q, k, v))
    dev = [x.cuda() for x in (q, k, v)]
    if bshd:
        dev = [x.transpose(1, 2).contiguous().transpose(1, 2) for x in dev]
    return (q, k, v), dev


def _exact(q, k, v, causal, wl):
    import torch
    B, H, S, D = q.shape
    group = H // k.shape[1]
    kk, vv = (x.double().repeat_interleave(group, dim=1) for x in (k, v))
    s = q.double() @ kk.transpose(2, 3).contiguous() / D ** 0.5
    i, j = torch.arange(S)[:, None], torch.arange(S)[None, :]
    if causal:
        s.masked_fill_(j > i, -np.inf)
    if wl >= 0:
        s.masked_fill_(j < i - wl, -np.inf)
    return torch.softmax(s, dim=-1) @ vv, torch.logsumexp(s, dim=-1)


@pytest.mark.parametrize("B,H,Hk,S,D,dtype,causal,wl,bshd,growth", CASES)
def test_reference_point_moves(forward, B, H, Hk, S, D, dtype, causal, wl, bshd, growth):
    import torch
    (q, k, v), (dq, dk, dv) = _inputs(B, H, Hk, S, D, dtype, growth, bshd, 31 + S + D)
    o, lse = forward(dq, dk, dv, causal=causal, window_left=wl, exact_first_rows=True)
    torch.cuda.synchronize()
    heads = slice(0, 2 * (H // Hk)), slice(0, 2)                      # (the first and last batch's first heads are enough)
    for b in {0, B - 1}:
        want, want_lse = _exact(q[b:b + 1, heads[0]], k[b:b + 1, heads[1]], v[b:b + 1, heads[1]], causal, wl)
        got = o[b:b + 1, heads[0]].cpu().double()
        u = 2.0 ** -8 if dtype == "bf16" else 2.0 ** -11
        assert bool(torch.isfinite(got).all())
        assert float((got - want).norm() / want.norm()) <= 1.5 * u
        assert float((got - want).abs().max()) <= 4 * u * float(v.abs().max())
        # fp32 sums of products of |q k| up to the largest score, 2^-24 each of D terms at most
        bound = 2.0 ** -24 * D * float(want_lse.abs().max()) + 1e-5
        assert float((lse[b:b + 1, heads[0]].cpu().double() - want_lse).abs().max()) <= bound


@pytest.mark.parametrize("S,D", [(512, 64), (512, 128), (500, 64), (500, 128)])
def test_nan_key_reaches_only_the_rows_that_see_it(forward, S, D):
    """A NaN in key 300 of a causal problem: rows from 300 on are NaN, the others what they are without it."""
    import torch
    _, (q, k, v) = _inputs(1, 2, 2, S, D, "fp16", 0.02, False, 77)
    clean, clean_lse = forward(q, k, v, causal=True)
    k = k.clone()
    k[:, :, 300, 5] = float("nan")
    o, lse = forward(q, k, v, causal=True)
    torch.cuda.synchronize()
    assert bool(torch.isnan(o[:, :, 300:]).all())
    assert torch.equal(o[:, :, :300], clean[:, :, :300])
    assert torch.equal(lse[:, :, :300], clean_lse[:, :, :300])


@pytest.mark.parametrize("B,H,Hk,S,Sk,D,dtype,causal,wl,bshd,splits", [
    (1, 2, 2, 1024, 1024, 64, "fp16", False, -1, False, 1),
    (1, 2, 2, 1024, 1024, 64, "fp16", True, -1, True, 1),
    (2, 16, 16, 2048, 2048, 128, "bf16", True, -1, False, 1),          # eight-wave workgroups
    (1, 2, 2, 1000, 1000, 128, "fp16", True, -1, False, 1),            # general kernels
    (1, 2, 2, 1000, 1000, 64, "bf16", False, -1, True, 1),
    (1, 64, 64, 2048, 2048, 64, "fp16", True, 700, False, 1),
    (1, 8, 1, 40, 3000, 128, "fp16", True, -1, True, 1),               # rows of several heads in one wave
    (1, 8, 2, 200, 5000, 64, "bf16", True, -1, True, 4),               # key splits
])
def test_rows_do_not_depend_on_each_other(forward, B, H, Hk, S, Sk, D, dtype, causal, wl, bshd, splits):
    """A query forty times as large moves its own reference point in many tiles (and sends its wave through the loop that takes
    maxima); every other row keeps its bits."""
    import torch
    g = torch.Generator().manual_seed(5 + S + D)
    dt = torch.bfloat16 if dtype == "bf16" else torch.float16
    q, k, v = (torch.randn((B, n, s, D), generator=g).to(dt).cuda() for n, s in ((H, S), (Hk, Sk), (Hk, Sk)))
    if bshd:
        q, k, v = (x.transpose(1, 2).contiguous().transpose(1, 2) for x in (q, k, v))
    kw = dict(causal=causal, window_left=wl, splits=splits, exact_first_rows=True)
    clean, clean_lse = forward(q, k, v, **kw)
    large = torch.arange(S) % 32 == 13
    large_heads = torch.arange(H) % 2 == 0
    q2 = q.clone(memory_format=torch.preserve_format)
    rows = (large_heads[:, None] & large[None, :]).cuda()
    q2[:, rows] = q2[:, rows] * 40
    o, lse = forward(q2, k, v, **kw)
    torch.cuda.synchronize()
    assert not torch.equal(o[:, rows], clean[:, rows])
    assert torch.equal(o[:, ~rows], clean[:, ~rows])
    assert torch.equal(lse[:, ~rows], clean_lse[:, ~rows])


@pytest.mark.parametrize("S,D,dtype,sigma,bound", [(2048, 128, "fp16", 4.0, 2.70e-4), (2048, 64, "bf16", 8.0, 1.97e-3), (2000, 64, "fp16", 4.0, 2.70e-4)])
def test_a_row_that_one_key_carries_has_its_weight_exact(forward, S, D, dtype, sigma, bound):
    """Sharp scores: the key that carries a row mostly has a weight of exactly 1, its own score being the reference point; a point
    that lags further behind rounds that weight too.  The bounds lie between the error of a point that lags by up to 2^8
    (2.60e-4 and 1.93e-3 of the outputs' norm against 64 bits) and by up to 2^12 (2.77e-4 and 1.98e-3)."""
    import torch
    g = torch.Generator().manual_seed(8)
    dt = torch.bfloat16 if dtype == "bf16" else torch.float16
    q, k, v = (torch.randn((1, 4, S, D), generator=g) for _ in range(3))
    q, k, v = (q * sigma).to(dt), k.to(dt), v.to(dt)
    o, _ = forward(q.cuda(), k.cuda(), v.cuda(), causal=True, exact_first_rows=True)
    want, _ = _exact(q, k, v, True, -1)
    assert float((o.cpu().double() - want).norm() / want.norm()) <= bound
