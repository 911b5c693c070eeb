"""Keys that a query does not see leave no trace in its output: the rows that take the verifier's arithmetic multiply every key of
the first thirty-two, seen or not, so infinities and NaN in V behind a row must not reach it (0 * inf would).  The rows in front of
the planted keys keep the bits of a run without them; the windowed rows past them as well.  In the items of a launch that fills the
chip (regular and general lengths), in workgroups beside a short launch, and with a few earlier keys."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape,S_kv", [((8, 32, 512, 64), 512), ((8, 32, 500, 128), 500), ((1, 2, 128, 64), 128), ((1, 2, 90, 128), 97),
                                        ((8, 64, 256, 128), 256), ((8, 40, 300, 64), 309)])
@pytest.mark.parametrize("window", [-1, 5])
def test_unseen_values_leave_no_trace(fa, dtype, shape, S_kv, window):
    B, H, S, D = shape
    g = torch.Generator(device="cuda").manual_seed(S + D)
    q = torch.randn(B, H, S, D, device="cuda", generator=g).to(dtype)
    k, v = (torch.randn(B, H, S_kv, D, device="cuda", generator=g).to(dtype) for _ in range(2))
    clean, lse = fa.flash_attention_forward(q, k, v, causal=True, window_left=window)
    planted = v.clone()
    planted[:, :, 13] = float("inf")
    planted[:, :, 17] = float("nan")
    got, lse2 = fa.flash_attention_forward(q, k, planted, causal=True, window_left=window)
    pos = torch.arange(S, device="cuda") + S_kv - S
    unseen = pos < 13
    if window >= 0:
        unseen |= (pos > 17 + window) & (pos < 32)
    assert torch.equal(got[:, :, unseen], clean[:, :, unseen])
    assert torch.equal(lse, lse2)
    assert not torch.isfinite(got[:, :, (pos >= 13) & (pos <= 13 + (window if window >= 0 else 18))]).any()
