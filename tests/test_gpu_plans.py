"""What the binding keeps per combination of shapes, strides and options: a call that finds an entry gives what the first
one gave, for other tensors, other strides and other options, and what was refused stays refused."""
import pytest

pytestmark = pytest.mark.gpu


def _inputs(torch, seed, bshd, B=2, H=4, Hk=2, S=200, D=64):
    g = torch.Generator(device="cuda").manual_seed(seed)
    t = [torch.randn((B, S, h, D) if bshd else (B, h, S, D), device="cuda", generator=g).half() for h in (H, Hk, Hk, H)]
    return [x.transpose(1, 2) for x in t] if bshd else t


@pytest.mark.parametrize("bshd", [False, True])
@pytest.mark.parametrize("kw", [dict(), dict(causal=True), dict(causal=True, window_left=40), dict(causal=True, splits=3),
                                dict(splits="auto", return_lse=False), dict(dropout_prob=0.2, seed=5), dict(softmax_scale=0.3), "slopes"])
def test_second_call_equals_the_first(fa, kw, bshd):
    import torch
    results = []
    for kept in (False, True):
        fa._plans.clear()
        if kept:            # entries of this shape made from other tensors (and, beside them, of other options and strides)
            for s, other in ((11, bshd), (12, not bshd)):
                q, k, v, do = _inputs(torch, s, other)
                for o in (dict(), dict(causal=True), dict(softmax_scale=0.5), dict() if kw == "slopes" else kw):
                    fa.flash_attention_forward(q, k, v, **o)
                if kw == "slopes":
                    fa.flash_attention_forward(q, k, v, alibi_slopes=torch.full((4,), 3.0, device="cuda"))
        q, k, v, do = _inputs(torch, 1, bshd)
        o = dict(alibi_slopes=torch.tensor([0.5, 0.25, 0.1, 0.0], device="cuda")) if kw == "slopes" else kw
        got = fa.flash_attention_forward(q, k, v, **o)
        out = list(got) if isinstance(got, tuple) else [got]
        o = {n: x for n, x in o.items() if n not in ("splits", "return_lse")}
        fwd, lse = fa.flash_attention_forward(q, k, v, exact_first_rows=True, **o)
        for _ in range(2):
            out += fa.flash_attention_backward(q, k, v, fwd, lse, do, **o)
        torch.cuda.synchronize()
        assert out[0].stride() == q.stride() and out[-1].stride() == v.stride()
        results.append(out)
    for a, b in zip(*results):
        assert a.stride() == b.stride()
        assert torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8))


def test_seeds_share_an_entry(fa):
    """A training with dropout has another seed every step: one entry for the forward and one for the backward pass serve
    them all, each with its own mask."""
    import torch
    q, k, v, do = _inputs(torch, 3, False)
    results = []
    for kept in (False, True):
        fa._plans.clear()
        for seed in (7, 0, (1 << 64) - 1, 8):
            if not kept:
                fa._plans.clear()
            kw = dict(dropout_prob=0.2, seed=seed)
            o, lse = fa.flash_attention_forward(q, k, v, exact_first_rows=True, **kw)
            results.append((o,) + fa.flash_attention_backward(q, k, v, o, lse, do, **kw))
    assert len(fa._plans) == 2
    torch.cuda.synchronize()
    for a, b in zip(results[:4], results[4:]):
        assert all(torch.equal(x.view(torch.int16), y.view(torch.int16)) for x, y in zip(a, b))
    assert not any(torch.equal(results[0][0], r[0]) for r in results[1:4])


def test_entries_hold_no_address(fa):
    import ctypes
    import torch
    fa._plans.clear()
    q, k, v, do = _inputs(torch, 5, True)
    slopes = torch.tensor([0.5, 0.25, 0.1, 0.0], device="cuda")
    o, lse = fa.flash_attention_forward(q, k, v, exact_first_rows=True, splits=3, alibi_slopes=slopes)
    fa.flash_attention_backward(q, k, v, o, lse, do, alibi_slopes=slopes)
    assert len(fa._plans) == 2
    for entry in fa._plans.values():
        kind = fa.FaFwdParams if len(entry[0]) == ctypes.sizeof(fa.FaFwdParams) else fa.FaBwdParams
        block = kind.from_buffer_copy(entry[0])
        assert [n for n, t in kind._fields_ if t is ctypes.c_void_p and getattr(block, n)] == []


def test_backward_with_an_entry_when_memory_is_short(fa, monkeypatch):
    """Room for the gradients and the small workspace, or for the kept entry's workspace alone: the call takes the smaller
    workspace, as it does without an entry.  (The limit is counted here; the device has memory enough.)"""
    import torch
    import weakref
    q, k, v, do = _inputs(torch, 4, False, B=1, H=8, Hk=8, S=512)
    o, lse = fa.flash_attention_forward(q, k, v, exact_first_rows=True)
    fa._plans.clear()
    want = fa.flash_attention_backward(q, k, v, o, lse, do)
    (_, total, _, _), = fa._plans.values()
    limit, used = total + (1 << 20), [0]
    assert total > (2 << 20) and 3 * q.numel() * 2 > (1 << 20)

    def counted(make):
        def wrapper(*args, **kw):
            t = make(*args, **kw)
            n = t.numel() * t.element_size()
            if used[0] + n > limit:
                raise torch.cuda.OutOfMemoryError("limit of this test")
            used[0] += n
            weakref.finalize(t, lambda: used.__setitem__(0, used[0] - n))
            return t
        return wrapper

    got = []
    for kept in (False, True):
        if not kept:
            plan = dict(fa._plans)
            fa._plans.clear()
        with monkeypatch.context() as m:
            m.setattr(torch, "empty", counted(torch.empty))
            m.setattr(torch, "empty_like", counted(torch.empty_like))
            got.append([x.clone() for x in fa.flash_attention_backward(q, k, v, o, lse, do)])
        fa._plans.update(plan)
    for a, b, w in zip(*got, want):
        assert torch.equal(a, b) and (a.float() - w.float()).norm() <= 2e-3 * w.float().norm()      # (each is within 1e-3 of the exact gradients)


def test_what_was_refused_stays_refused(fa):
    import torch
    q, k, v, _ = _inputs(torch, 1, False)
    fa.flash_attention_forward(q, k, v, causal=True, window_left=1, seed=1)
    for bad in (dict(window_left=1.0), dict(seed=1.0)):
        with pytest.raises(TypeError):
            fa.flash_attention_forward(q, k, v, **{**dict(causal=True, window_left=1, seed=1), **bad})
    scale = torch.tensor(0.25)
    a = fa.flash_attention_forward(q, k, v, softmax_scale=scale, return_lse=False).clone()
    scale.fill_(0.5)        # the same object with another value
    b = fa.flash_attention_forward(q, k, v, softmax_scale=scale, return_lse=False)
    assert torch.equal(b, fa.flash_attention_forward(q, k, v, softmax_scale=0.5, return_lse=False)) and not torch.equal(a, b)
    with pytest.raises(ValueError):
        fa.flash_attention_forward(q, k.cpu(), v)
    shifted = torch.empty(q.numel() + 8, dtype=q.dtype, device="cuda")[1:1 + q.numel()].view(q.shape)      # 2 bytes off
    with pytest.raises(fa.FaError):
        fa.flash_attention_forward(shifted, k, v, causal=True, window_left=1, seed=1)


def test_a_missing_native_part_is_said_on_the_first_call(fa, monkeypatch):
    import torch
    q = torch.randn((1, 2, 72, 64), device="cuda").half()
    monkeypatch.setattr(fa, "_native_module", None)
    monkeypatch.setattr(fa, "TORCH_LIB_PATH", "/nowhere/_fa_torch.so")
    with pytest.raises(RuntimeError, match="is missing"):
        fa.flash_attention_forward(q, q, q, causal=True)
    monkeypatch.undo()
    fa.flash_attention_forward(q, q, q, causal=True)
