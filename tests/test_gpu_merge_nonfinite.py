"""The merge of key splits where a part holds an infinity -- only parts that carry weight reach the result -- and where the
logsumexps are far from zero."""
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(1, 4, 2, 1, 704, 64), (2, 4, 4, 3, 704, 128),          # the decoding kernel
          (1, 4, 2, 200, 704, 64), (1, 2, 2, 200, 704, 128)]      # 128-row blocks


def _inputs(torch, B, H, Hk, S, Skv, D):
    g = torch.Generator(device="cuda").manual_seed(9)
    q = torch.randn((B, H, S, D), device="cuda", generator=g).half()
    k, v = (torch.randn((B, Hk, Skv, D), device="cuda", generator=g).half() for _ in range(2))
    return q, k, v


@pytest.mark.parametrize("splits", [3, 8, 11])        # a last batch of eight parts with five, no and five free places
@pytest.mark.parametrize("B,H,Hk,S,Skv,D", SHAPES)
def test_infinite_value_in_the_last_split(fa, B, H, Hk, S, Skv, D, splits):
    import torch
    q, k, v = _inputs(torch, B, H, Hk, S, Skv, D)
    want, lse_want = fa.flash_attention_forward(q, k, v, splits=splits)
    v[:, :, -1, 5] = float("inf")
    got, lse = fa.flash_attention_forward(q, k, v, splits=splits)
    torch.cuda.synchronize()
    assert bool((got[..., 5] == float("inf")).all())
    got[..., 5] = want[..., 5]
    assert torch.equal(got, want) and torch.equal(lse, lse_want)


@pytest.mark.parametrize("splits", [3, 8, 11])
@pytest.mark.parametrize("B,H,Hk,S,Skv,D", SHAPES)
def test_infinite_value_in_a_split_without_weight(fa, B, H, Hk, S, Skv, D, splits):
    """The last key's score is two thousand above all others: every other split's weight is exactly zero, and the result
    the last key's value, but for one rounding of the probability and one of the output to fp16 (2^-11 each)."""
    import torch
    q, k, v = _inputs(torch, B, H, Hk, S, Skv, D)
    q[..., 3] = 8.0
    k[:, :, -1, 3] = 2000.0 * D ** 0.5 / 8.0
    v[:, :, 7, 5] = float("inf")
    got, lse = fa.flash_attention_forward(q, k, v, splits=splits)
    torch.cuda.synchronize()
    want = v[:, :, -1:].repeat_interleave(H // Hk, 1).float()
    assert bool(((got.float() - want).abs() <= 2.0 ** -9 * want.abs() + 1e-6).all()) and bool(torch.isfinite(lse).all())


@pytest.mark.parametrize("sign", [1.0, -1.0])
@pytest.mark.parametrize("B,H,Hk,S,Skv,D", SHAPES)
def test_logsumexps_of_any_size(fa, B, H, Hk, S, Skv, D, sign):
    """All scores alike, a power of two of about 1e32 or its negative (exact in fp32, and so is the difference of two of
    them): the values, alike for all keys of a head, come back as they are."""
    import torch
    q, k, v = _inputs(torch, B, H, Hk, S, Skv, D)
    q.fill_(8.0)
    k.fill_(8.0 * sign)
    v.copy_(v[:, :, :1].expand_as(v).clone())
    for splits in (3, 11):
        got, lse = fa.flash_attention_forward(q, k, v, softmax_scale=2.0 ** 95, splits=splits)
        torch.cuda.synchronize()
        want = v[:, :, :1].repeat_interleave(H // Hk, 1).expand_as(got).float()
        assert bool(((got.float() - want).abs() <= 2.0 ** -10 * want.abs()).all())
        assert bool((lse == sign * 64.0 * D * 2.0 ** 95).all())


@pytest.mark.parametrize("B,H,Hk,S,Skv,D", SHAPES)
def test_logsumexps_that_overflow(fa, B, H, Hk, S, Skv, D):
    """Scaled scores of -2.9e38, a number in fp32 but not once multiplied by log2(e): the probabilities are infinite, the
    rows NaN without splits, and NaN, not an empty row, with them."""
    import torch
    q, k, v = _inputs(torch, B, H, Hk, S, Skv, D)
    q.fill_(8.0)
    k.fill_(-8.0)
    for splits in (1, 3, 11):
        got, lse = fa.flash_attention_forward(q, k, v, softmax_scale=2.9e38 / (64.0 * D), splits=splits)
        torch.cuda.synchronize()
        assert bool(torch.isnan(got).all()) and not bool(torch.isfinite(lse).any()) and not bool((lse == float("-inf")).any())


@pytest.mark.parametrize("splits", [1, 3, 8, 11])
@pytest.mark.parametrize("B,H,Hk,S,Skv,D", SHAPES + [(8, 16, 4, 200, 704, 64), (8, 16, 16, 200, 704, 128)])       # (128-row blocks without splits too)
def test_a_nan_is_not_lost(fa, B, H, Hk, S, Skv, D, splits):
    """A NaN in the last key of one head, in one split: that head's rows, which all see it, and their logsumexps are NaN however the
    keys are split; the other heads keep their bits."""
    import torch
    q, k, v = _inputs(torch, B, H, Hk, S, Skv, D)
    want, lse_want = fa.flash_attention_forward(q, k, v, splits=splits)
    k[0, 0, -1, 5] = float("nan")
    got, lse = fa.flash_attention_forward(q, k, v, splits=splits)
    torch.cuda.synchronize()
    group = H // Hk
    assert bool(torch.isnan(got[0, :group]).all()) and bool(torch.isnan(lse[0, :group]).all())
    for a, b in ((got, want), (lse, lse_want)):
        assert torch.equal(a[0, group:], b[0, group:]) and torch.equal(a[1:], b[1:])
