"""The decoding kernel (at most 32 query rows per K/V head) at the edges of its pieces, row blocks and key splits, against
the oracle on the last S rows of the square problem; the tolerances are the suite's (tests/parity_util.py)."""
import numpy as np
import pytest

from parity_util import assert_within, errors, from_torch, make_inputs, to_torch
from test_gpu_parity_decode import oracle_rect

pytestmark = pytest.mark.gpu

CASES = [
    # B, H, Hk, S, Skv, D, dtype, causal, wl, alibi, splits: rows per K/V head = H / Hk * S, pieces of 32 (D = 128) / 64 keys
    (1, 2, 2, 1, 1, 128, 0, False, -1, False, 1),          # one key
    (2, 2, 2, 1, 33, 64, 0, True, -1, False, 1),           # less than a piece
    (1, 4, 4, 1, 128, 128, 1, True, -1, False, 2),         # whole pieces, one for every wave
    (1, 4, 2, 8, 129, 128, 0, True, -1, False, 3),         # sixteen rows; one key in the last piece
    (1, 17, 1, 1, 300, 64, 0, True, -1, False, 2),         # seventeen rows: the second row block holds one
    (2, 16, 4, 8, 1000, 128, 1, True, -1, False, "auto"),  # thirty-two rows, ragged
    (1, 8, 1, 4, 2049, 64, 0, True, 64, False, 5),         # rows of a group see different windows; splits without any piece
    (1, 8, 8, 3, 700, 128, 0, True, 100, True, 11),        # more than eight partial results per row; ALiBi
    (2, 8, 2, 2, 4100, 64, 1, False, -1, True, "auto"),    # no mask: keys behind the last query, on both sides of it
    (1, 6, 3, 5, 64, 128, 0, True, 0, False, 1),           # every row sees one key
    (64, 16, 16, 20, 70, 128, 1, False, -1, True, 1),      # short keys, many heads: left to the tile kernels
    (128, 32, 8, 5, 104, 128, 0, True, 50, False, "auto"), # the same with a group's rows in one block
]


@pytest.mark.parametrize("B,H,Hk,S,Skv,D,dtype,causal,wl,alibi,splits", CASES)
def test_decode_kernel(fa, oracle, B, H, Hk, S, Skv, D, dtype, causal, wl, alibi, splits):
    import torch
    q, _, _ = make_inputs(fa, (B, H, S, D), dtype, seed=2000 + S)
    _, k, v = make_inputs(fa, (B, Hk, Skv, D), dtype, seed=2001 + Skv)
    slopes = np.power(2.0, -8.0 / H * (np.arange(H) + 1)).astype(np.float32) if alibi else None
    o_ref, lse_ref = oracle_rect(oracle, q, k, v, dtype, causal, wl, -1, slopes)
    tq, tk, tv = (to_torch(x, dtype) for x in (q, k, v))
    ts = torch.from_numpy(slopes).cuda() if alibi else None
    for bshd in (False, True):
        if bshd:
            tq, tk, tv = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (tq, tk, tv))
        o, lse = fa.flash_attention_forward(tq, tk, tv, causal=causal, window_left=wl, alibi_slopes=ts, splits=splits)
        torch.cuda.synchronize()
        got = oracle.to_f32(from_torch(o.contiguous()), dtype)
        err = errors(got, oracle.to_f32(o_ref, dtype), lse.cpu().numpy(), lse_ref)
        print((B, H, Hk, S, Skv, D), dtype, causal, wl, alibi, splits, bshd, err)
        if wl == 0 and dtype == 0:      # |O| as large as the values: one ulp of the result instead (see test_gpu_parity.py)
            assert err["nonfinite"] == 0 and err["max_abs"] <= max(2e-3, 2.0 ** -10 * float(np.abs(got).max()))
        else:
            assert_within(err, dtype, f"S={S} Skv={Skv} splits={splits}")


def test_decode_kernel_with_streaming_loads(fa):
    """K and V of more than 128 MB take the instantiations that read them with the non-temporal hint."""
    import torch
    B, H, Hk, S, Skv, D = 2, 32, 32, 1, 4100, 128
    g = torch.Generator(device="cuda").manual_seed(5)
    q = torch.randn((B, H, S, D), device="cuda", generator=g).half()
    k, v = (torch.randn((B, Hk, Skv, D), device="cuda", generator=g).half() for _ in range(2))
    o, lse = fa.flash_attention_forward(q, k, v, causal=True, splits="auto")
    s = (q.float() * k.float()).sum(-1) / D ** 0.5                      # one query per head
    p = torch.softmax(s, dim=-1)
    ref = (p[..., None] * v.float()).sum(2, keepdim=True)
    assert float((o.float() - ref).abs().max()) <= 2e-3
    assert float((lse[..., 0] - torch.logsumexp(s, dim=-1)).abs().max()) <= 2e-3


def test_auto_splits_fit_the_static_scratch(fa):
    """splits="auto" through the static scratch: where the partial results of the fastest split count do not fit the
    32 MiB, the count that fills the device once is used, whose do."""
    import ctypes
    import torch
    B, H, Hk, S, Skv, D = 146, 64, 2, 1, 4000, 128
    L = fa.lib()
    p = fa.make_params(B, H, S, D, causal=True, n_kv_heads=Hk, S_kv=Skv)
    need = {}
    for name, splits in (("auto", L.fa_fwd_auto_splits), ("fill", L.fa_fwd_suggest_splits)):
        p.split_num = splits(ctypes.byref(p))
        need[name] = L.fa_fwd_workspace_bytes(ctypes.byref(p))
    assert need["auto"] > L.fa_fwd_static_scratch_bytes() >= need["fill"] > 0
    g = torch.Generator(device="cuda").manual_seed(6)
    q = torch.randn((B, H, S, D), device="cuda", generator=g, dtype=torch.float16)
    k, v = (torch.randn((B, Hk, Skv, D), device="cuda", generator=g, dtype=torch.float16) for _ in range(2))
    o = fa.flash_attention_forward(q, k, v, causal=True, splits="auto", static_scratch=True, return_lse=False)
    ref = fa.flash_attention_forward(q, k, v, causal=True, splits=p.split_num, return_lse=False)
    assert torch.equal(o, ref)
