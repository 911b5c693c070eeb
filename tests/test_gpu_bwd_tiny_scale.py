"""The backward pass at softmax scales so small that lse / scale leaves fp32's range, against attention's gradients in 64 bits.

Inputs of order one give weights that are all alike (dV is then the mean of dO over the queries that see the key, and dQ and dK,
of the order of the scale, are nothing in the storage type); bf16 inputs of order 1e18 give scores of order one and gradients to
compare.  Tolerance: P, dS and the results are rounded to the storage type, u = 2^-11 or 2^-8 at most per value, about u in the
2-norm: 2 u."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _exact(q, k, v, do, scale, causal):
    import torch
    q, k, v, do = (x.double().cpu() for x in (q, k, v, do))
    s = q @ k.transpose(2, 3).contiguous() * scale
    if causal:
        n = q.shape[2]
        s.masked_fill_(torch.arange(n)[None, :] > torch.arange(n)[:, None], -np.inf)
    p = torch.softmax(s, dim=-1)
    dp = do @ v.transpose(2, 3).contiguous()
    ds = p * (dp - (p * dp).sum(-1, keepdim=True))
    return ds @ k * scale, ds.transpose(2, 3).contiguous() @ q * scale, p.transpose(2, 3).contiguous() @ do


@pytest.mark.parametrize("five", [True, False])
@pytest.mark.parametrize("S,D,dtype,causal,bshd,scale,size", [
    (1024, 64, "fp16", True, False, 1e-38, 1.0),
    (1024, 128, "fp16", False, True, 1e-40, 1.0),
    (1024, 128, "bf16", True, False, 3e-38, 1.0),
    (1000, 64, "bf16", True, False, 1.4e-45, 1.0),            # the smallest positive number; general kernels
    (1000, 64, "bf16", False, True, 1e-38, 1.5e18),
    (1024, 128, "bf16", True, False, 1e-38, 1.5e18),
    (512, 64, "bf16", True, False, 4e-32, 8e14),              # (below the rule's line)
    (512, 64, "bf16", True, False, 1e-30, 1.5e14),            # (above it)
])
def test_tiny_scales(fa, S, D, dtype, causal, bshd, scale, size, five):
    import torch
    g = torch.Generator().manual_seed(3 + S + D)
    dt = torch.bfloat16 if dtype == "bf16" else torch.float16
    q, k, v, do = (torch.randn((1, 2, S, D), generator=g) for _ in range(4))
    q, k, v, do = (x.to(dt).cuda() for x in (q * size, k * size, v, do))
    if bshd:
        q, k, v, do = (x.transpose(1, 2).contiguous().transpose(1, 2) for x in (q, k, v, do))
    kw = dict(causal=causal, softmax_scale=scale)
    o, lse = fa.flash_attention_forward(q, k, v, exact_first_rows=True, **kw)
    got = fa.flash_attention_backward(q, k, v, o, lse, do, five_products=five, **kw)
    torch.cuda.synchronize()
    want = _exact(q, k, v, do, float(np.float32(scale)), causal)
    u = 2.0 ** -8 if dtype == "bf16" else 2.0 ** -11
    for name, a, b in zip(("dQ", "dK", "dV"), got, want):
        a = a.double().cpu()
        assert bool(torch.isfinite(a).all()), name
        if name == "dV" or size > 1.0:
            assert float((a - b).norm() / b.norm()) <= 2 * u, name
        else:
            assert float((a - b).abs().max()) <= 1e-30, name
