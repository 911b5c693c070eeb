"""fa_fwd_auto_splits for chunks of queries behind a cache (the tile kernels): counts the library can run, the filling
count where the rule does not apply, and results at the edges of the rule against the oracle."""
import ctypes

import pytest

from parity_util import assert_within, errors, from_torch, make_inputs, to_torch
from test_gpu_parity_decode import oracle_rect


def both(fa, B, H, Hk, S, Skv, D, causal=True, wl=-1):
    p = fa.make_params(B, H, S, D, causal=causal, window_left=wl, n_kv_heads=0 if Hk == H else Hk, S_kv=Skv)
    return fa.lib().fa_fwd_auto_splits(ctypes.byref(p)), fa.lib().fa_fwd_suggest_splits(ctypes.byref(p))


def test_auto_splits_of_chunks(fa):
    for B, H, Hk, S, Skv, D in ((1, 1, 1, 33, 34, 64), (1, 1, 1, 200, 100000, 128), (1, 4, 1, 64, 20000, 128), (2, 8, 8, 33, 700, 64),
                                (1, 32, 8, 500, 4596, 128), (4, 16, 16, 600, 3000, 128), (1, 511, 511, 100, 4000, 128)):
        auto, _ = both(fa, B, H, Hk, S, Skv, D)
        tiles = (Skv + 63) // 64
        assert auto == 1 or 3 * auto <= tiles, (B, H, Hk, S, Skv, D, auto)
    # just over one workgroup per compute unit, or per slot: not twice as many rounds for it
    assert both(fa, 1, 256, 256, 100, 3000, 128)[0] == 1 and both(fa, 1, 86, 86, 300, 3000, 128)[0] != 2
    # a window, as many keys as queries, and problems that fill the device: as before
    for B, H, Hk, S, Skv, D, wl in ((1, 8, 8, 300, 4000, 128, 500), (1, 8, 8, 512, 512, 128, -1), (1, 8, 8, 500, 400, 64, -1),
                                    (2, 64, 64, 512, 9000, 128, -1), (4, 64, 64, 1700, 9000, 128, -1)):
        auto, fill = both(fa, B, H, Hk, S, Skv, D, True, wl)
        assert auto == fill


def test_splits_of_windowed_chunks(fa):
    """Behind a left window no more splits than tiles that some block visits, counted here block by block."""
    for B, H, Hk, S, Skv, D, wl in ((1, 8, 8, 64, 32768, 128, 128), (1, 16, 4, 1000, 9000, 64, 256), (1, 32, 32, 300, 4000, 128, 512),
                                    (1, 4, 4, 128, 32768, 64, 4096), (1, 2, 1, 50, 5000, 128, 0), (2, 8, 8, 129, 8000, 64, 1),
                                    (1, 1, 1, 200, 3000, 128, 2999), (1, 8, 2, 33, 2000, 64, 700)):
        rows = 128 if (H // Hk) * S > 128 or H == Hk else S
        most = max((min(r + rows, S) - 1 + Skv - S) // 64 - max(0, r + Skv - S - wl) // 64 + 1 for r in range(0, S, rows))
        auto, fill = both(fa, B, H, Hk, S, Skv, D, True, wl)
        assert auto == fill and auto <= most + 1, (S, Skv, wl, auto, most)       # (+ 1: the rule's blocks may lie anywhere)
    # many rows, whose partial results cost more than the tiles: none; few: some
    assert both(fa, 1, 16, 4, 1000, 9000, 64, True, 256)[0] == 1 and both(fa, 1, 8, 8, 47, 3477, 128, True, 331)[0] > 3


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,Hk,S,Skv,D,dtype,causal", [
    (1, 2, 2, 33, 193, 64, 0, True),          # the smallest chunk, four tiles: one split
    (1, 4, 1, 65, 1601, 128, 1, True),        # three blocks in one K/V head, one key in the last tile
    (1, 2, 1, 200, 2000, 64, 0, False),       # no mask
    (2, 3, 3, 129, 1100, 128, 0, True),       # a last block of one row
])
def test_chunks_with_auto_splits(fa, oracle, B, H, Hk, S, Skv, D, dtype, causal):
    import torch
    q, _, _ = make_inputs(fa, (B, H, S, D), dtype, seed=3000 + S)
    _, k, v = make_inputs(fa, (B, Hk, Skv, D), dtype, seed=3001 + Skv)
    o_ref, lse_ref = oracle_rect(oracle, q, k, v, dtype, causal, -1, -1, None)
    o, lse = fa.flash_attention_forward(*(to_torch(x, dtype) for x in (q, k, v)), causal=causal, splits="auto")
    torch.cuda.synchronize()
    err = errors(oracle.to_f32(from_torch(o), dtype), oracle.to_f32(o_ref, dtype), lse.cpu().numpy(), lse_ref)
    assert_within(err, dtype, f"S={S} Skv={Skv} splits={both(fa, B, H, Hk, S, Skv, D, causal)[0]}")


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,Hk,S,Skv,D,dtype,wl,splits", [
    (1, 2, 2, 150, 1500, 64, 0, 100, 3),          # every block sees four or five of 24 tiles
    (1, 2, 1, 150, 1500, 128, 1, 40, 7),          # more splits than tiles: some shares hold nothing
    (1, 4, 1, 30, 2000, 128, 0, 300, 4),          # four heads' rows in one block
    (1, 2, 2, 256, 300, 64, 0, 0, 5),             # every row sees one key
    (1, 2, 2, 300, 310, 128, 0, 64, 4),           # the first rows' arithmetic (queries from position 10 on)
])
def test_windows_with_splits(fa, oracle, B, H, Hk, S, Skv, D, dtype, wl, splits):
    import torch
    q, _, _ = make_inputs(fa, (B, H, S, D), dtype, seed=4000 + S)
    _, k, v = make_inputs(fa, (B, Hk, Skv, D), dtype, seed=4001 + Skv)
    o_ref, lse_ref = oracle_rect(oracle, q, k, v, dtype, True, wl, -1, None)
    o, lse = fa.flash_attention_forward(*(to_torch(x, dtype) for x in (q, k, v)), causal=True, window_left=wl, splits=splits)
    torch.cuda.synchronize()
    got = oracle.to_f32(from_torch(o), dtype)
    err = errors(got, oracle.to_f32(o_ref, dtype), lse.cpu().numpy(), lse_ref)
    if wl == 0:                                   # |O| as large as the values: one ulp of the result
        assert err["nonfinite"] == 0 and err["max_abs"] <= max(2e-3, 2.0 ** -10 * abs(got).max())
    else:
        assert_within(err, dtype, f"S={S} Skv={Skv} wl={wl} splits={splits}")
