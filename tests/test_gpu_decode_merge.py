"""Key splits that the decoding kernel merges itself, against the same call without splits: the split counts around its batches
of eight and its groups, the fewest and the most rows, empty splits; the counters are left as they were found, on several streams
and in replayed graphs."""
import pytest

pytestmark = pytest.mark.gpu


def _inputs(torch, seed, B, H, Hk, S, Sk, D, dtype="float16"):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.randn((B, h, n, D), device="cuda", generator=g).to(getattr(torch, dtype)) for h, n in ((H, S), (Hk, Sk), (Hk, Sk))]


def _close(torch, a, b, dtype):
    # the same weights in another order of fp32 sums, then one rounding: one place of the storage type of the larger values
    tol = 2.0 ** -9 if dtype == "float16" else 2.0 ** -6
    assert float((a.float() - b.float()).abs().max()) <= tol * max(1.0, float(b.float().abs().max()))


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("B,H,Hk,S,Sk,D,splits,window", [
    (1, 4, 4, 1, 1000, 64, 2, -1), (1, 8, 2, 1, 1003, 128, 8, -1), (2, 8, 1, 1, 2000, 128, 7, -1), (1, 1, 1, 1, 5000, 64, 9, -1), (1, 2, 2, 1, 5000, 128, 33, -1),
    (1, 1, 1, 1, 20000, 64, 64, -1), (1, 1, 1, 2, 10000, 64, 60, -1), (3, 4, 2, 3, 700, 64, 5, -1), (1, 16, 1, 1, 900, 128, 4, -1), (2, 30, 2, 2, 600, 64, 4, -1),
    (1, 32, 1, 1, 500, 128, 2, -1), (1, 4, 2, 1, 3000, 128, 12, 100), (256, 2, 2, 1, 300, 64, 2, -1), (257, 2, 2, 1, 300, 64, 2, -1)])
def test_splits_merged_inside(fa, dtype, B, H, Hk, S, Sk, D, splits, window):
    import torch
    q, k, v = _inputs(torch, Sk + splits, B, H, Hk, S, Sk, D, dtype)
    kw = dict(causal=True, window_left=window)
    o, lse = fa.flash_attention_forward(q, k, v, splits=splits, **kw)
    again, lse2 = fa.flash_attention_forward(q, k, v, splits=splits, **kw)
    ref, lse_ref = fa.flash_attention_forward(q, k, v, splits=1, **kw)
    assert torch.equal(o, again) and torch.equal(lse, lse2)
    _close(torch, o, ref, dtype)
    assert float((lse - lse_ref).abs().max()) <= 1e-4


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("B,H,Hk,S,Sk,D,splits", [
    (1, 8, 2, 1, 1003, 128, 7), (2, 4, 4, 2, 2000, 64, 8), (1, 14, 2, 1, 1200, 128, 9), (1, 10, 2, 1, 2000, 128, 12), (2, 9, 1, 1, 2000, 64, 14),
    (1, 8, 2, 1, 2100, 128, 16), (1, 6, 2, 1, 4000, 128, 20), (1, 2, 1, 3, 4000, 64, 20), (3, 7, 7, 1, 2200, 64, 17), (1, 1, 1, 1, 5000, 128, 63),
    (1, 2, 1, 1, 9000, 64, 60), (2, 1, 1, 1, 9000, 64, 66), (1, 1, 1, 1, 9000, 64, 128)])
def test_bits_do_not_depend_on_which_kernel_merges(fa, dtype, B, H, Hk, S, Sk, D, splits):
    """The same call with a counter set, its splits merged in the decoding kernel, and without one (hipStreamPerThread has none), merged
    by the second kernel: one batch of parts, several that threads take in turn, and up to eight groups of them."""
    import ctypes
    import torch
    q, k, v = _inputs(torch, Sk + splits, B, H, Hk, S, Sk, D, dtype)
    results = []
    for stream in (torch.cuda.current_stream().cuda_stream, 2):
        o, lse = torch.full_like(q, float("nan")), torch.full((B, H, S), float("nan"), device="cuda")
        p = fa.make_params(B, H, S, D, q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr(), causal=True, n_kv_heads=0 if Hk == H else Hk,
                           S_kv=Sk, split_num=splits, dtype=fa.FA_DTYPE_BF16 if dtype == "bfloat16" else fa.FA_DTYPE_F16)
        workspace = torch.empty(fa.lib().fa_fwd_workspace_bytes(ctypes.byref(p)), dtype=torch.uint8, device="cuda")
        p.workspace, p.workspace_bytes = workspace.data_ptr(), workspace.numel()
        torch.cuda.synchronize()
        assert fa.lib().fa_fwd(ctypes.byref(p), ctypes.c_void_p(stream)) == fa.FA_OK
        torch.cuda.synchronize()
        assert not o.isnan().any() and not lse.isnan().any()
        results.append((o.view(torch.int16), lse.view(torch.int32)))
    assert torch.equal(results[0][0], results[1][0]) and torch.equal(results[0][1], results[1][1])


def test_streams_and_graphs(fa):
    """More streams than there are sets, launches of all of them in flight together, and a graph of more launches than there are
    sets for captured ones: every result is the first one's."""
    import torch
    calls = [_inputs(torch, s, *shape) for s, shape in enumerate([(1, 8, 2, 1, 1003, 128), (2, 4, 4, 1, 2000, 64), (1, 16, 1, 1, 900, 128)])]
    run = lambda c: fa.flash_attention_forward(*c, causal=True, splits=8, return_lse=False)
    ref = [fa.flash_attention_forward(*c, causal=True, splits=1, return_lse=False) for c in calls]
    streams = [torch.cuda.Stream() for _ in range(70)]
    torch.cuda.synchronize()
    outs = []
    for _ in range(3):
        for n, s in enumerate(streams):
            with torch.cuda.stream(s):
                outs.append((n % 3, run(calls[n % 3])))
    torch.cuda.synchronize()
    for n, o in outs:
        _close(torch, o, ref[n], "float16")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = [(n % 3, run(calls[n % 3])) for n in range(240)]
    for _ in range(4):
        for _, o in captured:
            o.fill_(float("nan"))
        graph.replay()
        eager = [run(c) for c in calls]
        torch.cuda.synchronize()
        for n, o in captured + list(enumerate(eager)):
            _close(torch, o, ref[n], "float16")
    import ctypes
    for s in streams:
        assert fa.lib().fa_release_work_queue(ctypes.c_void_p(s.cuda_stream)) == fa.FA_OK
