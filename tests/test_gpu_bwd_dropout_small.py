"""Backward with dropout in fp16 where dS lies in the storage type's subnormal range (small dO): P and dS carry the factor
1 / (1 - p) before they are rounded, so what rounding adds does not grow with it.

Tolerance: dS <= 2^-13 is rounded to a multiple of 2^-24, an error of 2^-24 / sqrt(12) per pair (r.m.s.).  An element of dK sums
such errors over the queries that see its key, weighted with scale * Q (unit variance), dQ over the keys its query sees, and
is rounded itself; larger values add a relative 2^-11 for dS and one for O in delta.  1.5 times the sum, in the 2-norm (at
p = 0.9 a factor of 10 behind the rounding exceeds it at least twice, at p = 0.5 a factor of 2 by a tenth)."""
import numpy as np
import pytest

from parity_util import from_torch, make_inputs, to_torch
from test_gpu_parity_bwd import oracle_bwd_general

pytestmark = pytest.mark.gpu

CASES = [
    # B, H, Hk, S, D, causal, bshd, p, sigma of dO, five products
    (1, 2, 2, 1024, 64, False, False, 0.5, 1e-4, True),
    (1, 2, 2, 1024, 64, False, True, 0.9, 1e-3, True),
    (1, 2, 1, 1024, 128, True, True, 0.9, 1e-3, True),
    (1, 2, 2, 1024, 128, False, False, 0.5, 1e-4, False),
    (1, 2, 2, 1000, 64, True, False, 0.9, 1e-4, False),       # general kernels
    (1, 2, 2, 1000, 128, False, True, 0.9, 1e-4, False),
]


@pytest.mark.parametrize("B,H,Hk,S,D,causal,bshd,p,sigma,five", CASES)
def test_small_gradients_keep_their_precision(fa, oracle, B, H, Hk, S, D, causal, bshd, p, sigma, five):
    import torch
    thr, seed = fa.lib().fa_dropout_threshold(p), 21
    q, _, _ = make_inputs(fa, (B, H, S, D), 0, seed=810 + S)
    do, _, _ = make_inputs(fa, (B, H, S, D), 0, seed=811 + S, sigma=sigma)
    _, k, v = make_inputs(fa, (B, Hk, S, D), 0, seed=812 + S)
    want = oracle_bwd_general(oracle, q, k, v, do, 0, causal, -1, -1, None, dropout=(thr, seed))
    tq, tk, tv, tdo = (to_torch(x, 0) for x in (q, k, v, do))
    if bshd:
        tq, tk, tv, tdo = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (tq, tk, tv, tdo))
    kw = dict(causal=causal, dropout_prob=p, seed=seed)
    o, lse = fa.flash_attention_forward(tq, tk, tv, exact_first_rows=True, **kw)
    got = fa.flash_attention_backward(tq, tk, tv, o, lse, tdo, five_products=five, **kw)
    torch.cuda.synchronize()
    step, pairs = 2.0 ** -24 / np.sqrt(12.0), S * (0.5 if causal else 1.0)
    for name, g, w, n in (("dQ", got[0], want[0], pairs), ("dK", got[1], want[1], pairs * H // Hk)):
        err = oracle.to_f32(from_torch(g.contiguous()), 0).astype(np.float64) - w
        rms, size = np.sqrt(np.mean(err ** 2)), np.sqrt(np.mean(w ** 2))
        bound = 1.5 * (np.hypot(step * np.sqrt(n / D), step) + 2 * 2.0 ** -11 * size)
        print((B, H, Hk, S, D), causal, bshd, p, sigma, five, name, "rms", rms, "bound", bound, "size", size, flush=True)
        assert rms <= bound, (name, rms, bound)
