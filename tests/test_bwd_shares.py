"""Equal shares of the key-owning backward kernel's work (fa_bwd_shared): the arithmetic on the host, and the gradients
on the GPU where walks are cut at the odd places."""
import os
import subprocess
import tempfile

import numpy as np
import pytest

from parity_util import from_torch, make_inputs, to_torch
from test_gpu_parity_bwd import check, grad_errors, oracle_bwd_general

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_shares_cover_every_walk_once():
    """tests/c/check_bwd_shares.c: the shares of the walks, the slots of their parts and the rule that adds them."""
    with tempfile.TemporaryDirectory() as tmp:
        exe = os.path.join(tmp, "check_bwd_shares")
        subprocess.run(["gcc", "-O2", "-Wall", "-Wextra", "-I", os.path.join(REPO, "flash-attn-rtx5060_amd", "csrc"),
                        os.path.join(REPO, "tests", "c", "check_bwd_shares.c"), "-o", exe], check=True)
        out = subprocess.run([exe], stdout=subprocess.PIPE, text=True)
    assert out.returncode == 0, out.stdout


def test_launches_fit_the_buffer_of_the_parts():
    """tests/c/check_bwd_share_slots.c: the shares of every launch against what fa_bwd_share_bytes sizes, for devices of
    other compute unit counts as well."""
    with tempfile.TemporaryDirectory() as tmp:
        exe = os.path.join(tmp, "check_bwd_share_slots")
        subprocess.run(["gcc", "-O2", "-Wall", "-Wextra", "-I", os.path.join(REPO, "flash-attn-rtx5060_amd", "csrc"),
                        os.path.join(REPO, "tests", "c", "check_bwd_share_slots.c"), "-o", exe], check=True)
        out = subprocess.run([exe], stdout=subprocess.PIPE, text=True)
    assert out.returncode == 0, out.stdout


def test_share_bytes_and_refusals(fa):
    import ctypes
    L = fa.lib()
    ok = dict(B=2, N=16, S=1024, d=128, n_kv_heads=4, q_ptr=0x1000, k_ptr=0x2000, v_ptr=0x3000, o_ptr=0x4000, do_ptr=0x5000, lse_ptr=0x6000,
              dq_ptr=0x7000, dk_ptr=0x8000, dv_ptr=0x9000, workspace_ptr=0xA000, workspace_bytes=1 << 30)
    p = fa.make_bwd_params(**ok)
    need = L.fa_bwd_share_bytes(ctypes.byref(p))
    # 8 K/V heads, four walks of 4 * 16 pairs each: 2048 pairs, a share for every compute unit
    assert need == 256 * 2 * 2 * 256 * 128 * 4
    assert L.fa_bwd_share_bytes(ctypes.byref(fa.make_bwd_params(**{**ok, "S": 128, "n_kv_heads": 16}))) == 0          # nothing to cut
    assert L.fa_bwd_share_bytes(ctypes.byref(fa.make_bwd_params(**{**ok, "S_kv": 2048}))) == 0      # no five-product form
    # head dimension 64, where the uncut launch has items of 128 keys, two workgroups to a compute unit: a longest walk of 16 pairs
    # of 128 keys each against shares of 2.5 or 5 pairs is not worth a cut, walks of 128 are
    for B, N, Nk, S, cut in ((1, 16, 16, 1024, 0), (4, 8, 8, 1024, 0), (5, 8, 8, 4096, 0), (1, 8, 8, 2048, 256), (1, 32, 8, 2048, 256)):
        q = fa.make_bwd_params(**{**ok, "B": B, "N": N, "n_kv_heads": Nk, "S": S, "d": 64, "causal": True, "workspace_bytes": 1 << 40})
        assert L.fa_bwd_share_bytes(ctypes.byref(q)) == cut * 2 * 2 * 256 * 64 * 4
    assert L.fa_bwd_shared(ctypes.byref(p), 0xB008, need, None) == fa.FA_ERR_WORKSPACE              # alignment
    assert L.fa_bwd_shared(ctypes.byref(p), 0xB000, need - 1, None) == fa.FA_ERR_WORKSPACE


CASES = [
    # B, H, Hk, S, D, dtype, causal, wl, wr, bshd, alibi, dropout: (heads * walks) pairs over as many shares as fit
    (1, 8, 1, 1000, 128, 0, True, -1, -1, True, False, 0.0),     # one K/V head, every walk cut several times, ragged
    (1, 8, 2, 1024, 64, 1, True, -1, -1, False, False, 0.0),     # strided kernels, no remainder
    (1, 4, 4, 1280, 128, 1, True, -1, -1, False, False, 0.0),    # contiguous layout: walks end inside and at the ends of shares
    (1, 2, 2, 1100, 64, 0, False, -1, -1, False, False, 0.0),    # no mask, ragged: the last block has 76 keys
    (2, 6, 2, 768, 128, 0, True, 300, -1, True, False, 0.0),     # window: walks of unequal lengths
    (1, 8, 2, 640, 128, 0, True, -1, -1, True, True, 0.0),       # ALiBi: a share begins in the middle of a group
    (1, 8, 4, 896, 64, 0, False, -1, -1, True, False, 0.2),      # dropout
]


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,Hk,S,D,dtype,causal,wl,wr,bshd,alibi,dropout", CASES)
def test_gradients_from_shares(fa, oracle, B, H, Hk, S, D, dtype, causal, wl, wr, bshd, alibi, dropout):
    import torch
    thr, seed = fa.lib().fa_dropout_threshold(dropout), 48
    q, _, _ = make_inputs(fa, (B, H, S, D), dtype, seed=720 + S)
    do, _, _ = make_inputs(fa, (B, H, S, D), dtype, seed=721 + S)
    _, k, v = make_inputs(fa, (B, Hk, S, D), dtype, seed=722 + S)
    slopes = (np.power(2.0, -8.0 / H * (np.arange(H) + 1))).astype(np.float32) if alibi else None
    refs = oracle_bwd_general(oracle, q, k, v, do, dtype, causal, wl, wr, slopes, **(dict(dropout=(thr, seed)) if thr else {}))
    tq, tk, tv, tdo = (to_torch(x, dtype) for x in (q, k, v, do))
    if bshd:
        tq, tk, tv, tdo = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (tq, tk, tv, tdo))
    kw = dict(causal=causal, window_left=wl, window_right=wr, alibi_slopes=None if slopes is None else torch.from_numpy(slopes).cuda(),
              dropout_prob=dropout, seed=seed)
    o, lse = fa.flash_attention_forward(tq, tk, tv, exact_first_rows=True, **kw)
    shared = fa.flash_attention_backward(tq, tk, tv, o, lse, tdo, poison_workspace=True, **kw)
    again = fa.flash_attention_backward(tq, tk, tv, o, lse, tdo, poison_workspace=True, **kw)
    whole = fa.flash_attention_backward(tq, tk, tv, o, lse, tdo, five_products=True, **kw)
    torch.cuda.synchronize()
    grow = 256.0 / (256 - thr)          # kept probabilities are multiplied by 1/(1-p), and so is every rounding error
    for name, got, rerun, want, one in zip(("dQ", "dK", "dV"), shared, again, refs, whole):
        err = grad_errors(oracle.to_f32(from_torch(got.contiguous()), dtype), want / grow)
        print((B, H, Hk, S, D), dtype, causal, wl, wr, bshd, alibi, dropout, name, err, flush=True)
        if thr == 0:
            check(err, dtype, name)
        same = torch.equal(got.contiguous().view(torch.int16), rerun.contiguous().view(torch.int16))
        assert same, name
        # against the walks in one piece: sums of the same products in another order (dQ: the same order), so at most one
        # rounding of the result apart nearly everywhere
        diff = float((got.float() - one.float()).norm() / one.float().norm())
        assert diff <= (2.0 ** -8 if dtype else 2.0 ** -11), (name, diff)
