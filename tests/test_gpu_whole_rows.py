"""The general 128-wide kernels write their results through LDS, whole rows at a time: every row that exists is written, and no other.
O lies in a larger buffer whose other bytes must stay as they were; lengths at the edges of a wave's 32 rows and a workgroup's 128 or
256, key splits (fp32 partial results), packed groups, rows that see no key, and items in front of and behind one with first rows.
Small problems as they are, which the kernel of 32-row blocks or the decoding kernel writes, and among copies of themselves."""
import pytest
import torch

from parity_util import among_others, copies_for_tiles

pytestmark = pytest.mark.gpu


def reference(q, k, v, causal, window):
    S, Sk, rep = q.shape[2], k.shape[2], q.shape[1] // k.shape[1]
    k, v = (x.float().repeat_interleave(rep, 1) for x in (k, v))
    s = torch.matmul(q.float(), k.transpose(2, 3).contiguous()) / q.shape[3] ** 0.5
    i, j = torch.arange(S, device="cuda")[:, None] + Sk - S, torch.arange(Sk, device="cuda")[None]
    seen = torch.ones_like(i + j, dtype=torch.bool)
    if causal:
        seen &= j <= i
    if window >= 0:
        seen &= i - j <= window
    s = s.masked_fill(~seen, float("-inf"))
    return torch.nan_to_num(torch.softmax(s, -1)) @ v


@pytest.mark.parametrize("tiles", [False, True], ids=["alone", "among_others"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,H,Hk,S,S_kv,causal,window,splits", [
    (1, 2, 2, 1, 300, False, -1, 1), (2, 3, 1, 31, 64, True, -1, 1), (2, 4, 2, 33, 200, True, -1, 3), (3, 40, 8, 97, 500, False, -1, 2),
    (2, 4, 4, 129, 129, True, -1, 1), (1, 8, 8, 255, 255, True, 40, 1), (8, 64, 64, 257, 257, True, -1, 1), (4, 64, 64, 500, 500, True, -1, 1),
    (2, 64, 64, 1100, 1100, True, -1, 1), (4, 64, 16, 300, 1200, True, -1, 1),                            # 256-row workgroups
    (1, 4, 4, 200, 90, True, -1, 1), (1, 4, 4, 200, 90, True, -1, 2), (1, 8, 2, 500, 2500, True, 300, 4), (1, 8, 2, 13, 2500, True, -1, 7)])
def test_rows_and_nothing_else(fa, dtype, tiles, B, H, Hk, S, S_kv, causal, window, splits):
    g = torch.Generator(device="cuda").manual_seed(S * 7 + S_kv)
    q = torch.randn(B, H, S, 128, device="cuda", generator=g).to(dtype)
    k, v = (torch.randn(B, Hk, S_kv, 128, device="cuda", generator=g).to(dtype) for _ in range(2))
    copies = copies_for_tiles(fa, q, k, causal=causal, window_left=window, splits=splits, exact_first_rows=True) if tiles else 1
    if tiles and copies == 1:
        return                     # (nothing else than alone)
    room = torch.full((B * copies, S + 2, H + 1, 136), 7.0, device="cuda", dtype=dtype)      # [B, S, H, D] with gaps everywhere
    out = room[:, 1:S + 1, :H, :128].transpose(1, 2)
    o, lse = fa.flash_attention_forward(*(among_others(t, copies) for t in (q, k, v)), causal=causal, window_left=window, splits=splits,
                                        exact_first_rows=True, out=out)
    ref = reference(q, k, v, causal, window)
    # probabilities and output are rounded to the storage type once each, everything else is fp32
    u = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    assert torch.equal(out[:B], out[-B:]) and (out[:B].float() - ref).abs().max().item() <= 2 * u * v.float().abs().max().item() + 1e-4
    out.fill_(7.0)
    assert torch.equal(room, torch.full_like(room, 7.0))
