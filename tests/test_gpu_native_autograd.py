"""The differentiable operator in C++ against the Python function that it stands in for: the same bits in both directions, on the
first call of a combination and on the ones that find its plan; what the Python function refuses or cannot do stays so."""
import pytest

pytestmark = pytest.mark.gpu


def _inputs(torch, seed, S, D, H, Hk, bshd, dtype):
    g = torch.Generator(device="cuda").manual_seed(seed)
    t = [torch.randn((2, S, h, D) if bshd else (2, h, S, D), device="cuda", generator=g).to(dtype) for h in (H, Hk, Hk, H)]
    t = [x.transpose(1, 2) for x in t] if bshd else t
    return [x.requires_grad_(True) for x in t[:3]] + [t[3]]


def _python(torch, fa, q, k, v, **opts):
    """The operator through the function in Python (a subclass of torch.Tensor takes that way)."""
    class Sub(torch.Tensor):
        pass
    return fa.flash_attention(q.as_subclass(Sub), k, v, **opts).as_subclass(torch.Tensor)


@pytest.mark.parametrize("S,D,H,Hk,bshd,dtype,kw", [
    (128, 64, 4, 4, False, "float16", {}), (200, 64, 4, 2, True, "float16", dict(causal=True)), (384, 128, 8, 2, True, "bfloat16", dict(causal=True, window_left=100)),
    (256, 64, 4, 4, True, "float16", dict(dropout_prob=0.2, seed=(1 << 64) - 3)), (128, 128, 4, 4, False, "bfloat16", dict(softmax_scale=1)),
    (128, 64, 4, 4, False, "float16", "slopes"), (1, 64, 4, 1, False, "float16", dict(causal=1))])
def test_bits_of_the_python_function(fa, S, D, H, Hk, bshd, dtype, kw):
    import torch
    if kw == "slopes":
        kw = dict(alibi_slopes=torch.tensor([0.5, 0.25, 0.1, 0.0], device="cuda"), causal=True)
    for seed in (1, 2, 3):
        q, k, v, do = _inputs(torch, seed, S, D, H, Hk, bshd, getattr(torch, dtype))
        for grad in (do, torch.ones((), device="cuda", dtype=do.dtype).expand(do.shape)):          # (the second has no strides of its own)
            o = fa.flash_attention(q, k, v, **kw)
            got = (o.detach(),) + torch.autograd.grad(o, (q, k, v), grad)
            p = _python(torch, fa, q, k, v, **kw)
            want = (p.detach(),) + torch.autograd.grad(p, (q, k, v), grad)
            assert "Python" not in type(o.grad_fn).__name__ and o.grad_fn is not None
            for a, b in zip(got, want):
                assert a.stride() == b.stride() and torch.equal(a.contiguous().view(torch.int16), b.contiguous().view(torch.int16))


def test_hooks_graphs_and_refusals(fa):
    import torch
    q, k, v, do = _inputs(torch, 5, 128, 64, 4, 4, False, torch.float16)
    packed, unpacked = [], []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.shape) or t, lambda t: unpacked.append(t.shape) or t):
        o = fa.flash_attention(q, k, v, causal=True)
    first = torch.autograd.grad(o, (q, k, v), do, retain_graph=True)
    assert len(packed) == 5 and len(unpacked) == 5
    again = torch.autograd.grad(o, (q, k, v), do)
    assert all(torch.equal(a, b) for a, b in zip(first, again))
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(o, (q,), do)
    with torch.no_grad():
        assert fa.flash_attention(q, k, v).grad_fn is None
    o = fa.flash_attention(q, k.detach(), v.detach())
    assert torch.autograd.grad(o, (q,), do)[0].shape == q.shape
    with pytest.raises(ValueError):
        fa.flash_attention(q, k.cpu(), v)
    with pytest.raises(ValueError):
        fa.flash_attention(q, k.bfloat16(), v)
    with pytest.raises(TypeError):
        fa.flash_attention(q, k, v, window_left=1.0)
    with pytest.raises(fa.FaError):
        fa.flash_attention(q, k, v, softmax_scale=-1.0)
    for too_large in (dict(softmax_scale=10 ** 400), dict(dropout_prob=10 ** 400)):
        with pytest.raises(OverflowError):
            fa.flash_attention(q, k, v, **too_large)
    fa.flash_attention(q, k, v, softmax_scale=0.5)
    shifted = torch.empty(q.numel() + 8, dtype=q.dtype, device="cuda")[1:1 + q.numel()].view(q.shape)       # 2 bytes off, a known combination
    with pytest.raises(fa.FaError):
        fa.flash_attention(shifted, k, v, softmax_scale=0.5)
    # a gradient that is 2 bytes off is found in the engine's thread
    o = fa.flash_attention(q, k, v, softmax_scale=0.5)
    torch.autograd.grad(o, (q, k, v), do, retain_graph=True)
    bad = torch.empty(do.numel() + 8, dtype=do.dtype, device="cuda")[1:1 + do.numel()].view(do.shape)
    with pytest.raises(fa.FaError):
        torch.autograd.grad(o, (q, k, v), bad)
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda x: fa.flash_attention(x, k, v))(torch.stack([q, q]))


def test_a_subclass_of_the_query_is_the_class_of_the_output(fa):
    """The first call of a combination, the ones from its plan, and those whose plan a plain tensor has made."""
    import torch

    class Sub(torch.Tensor):
        pass
    for n, plain_first in ((232, False), (248, True)):
        q, k, v, _ = (t.detach() for t in _inputs(torch, 8, n, 64, 4, 4, False, torch.float16))
        calls = [q, q] if plain_first else []
        for x in calls + [q.as_subclass(Sub)] * 3 + [torch.nn.Parameter(q)]:
            o, lse = fa.flash_attention_forward(x, k, v)
            assert type(o) is (Sub if type(x) is Sub else torch.Tensor) and type(lse) is torch.Tensor
            assert type(fa.flash_attention_forward(x, k.as_subclass(Sub), v, return_lse=False)) is type(o)
            assert type(fa.flash_attention(x, k, v)) is type(o)


@pytest.mark.filterwarnings("ignore::torch.jit.TracerWarning")
def test_ways_that_stay_with_the_python_function(fa, monkeypatch):
    """Forward mode, the transforms of torch.func and tracing never reach the function in C++ (which is made to fail here), compiled code
    gives what eager code does."""
    import torch
    import torch.autograd.forward_ad as forward_ad
    q, k, v, do = _inputs(torch, 9, 136, 64, 4, 4, False, torch.float16)
    o = fa.flash_attention(q, k, v)
    want = (o.detach(),) + torch.autograd.grad(o, (q, k, v), do)
    compiled = torch.compile(lambda *t: fa.flash_attention(*t) * 1, backend="eager")(q, k, v)
    got = (compiled.detach(),) + torch.autograd.grad(compiled, (q, k, v), do)
    assert all(torch.equal(a, b) for a, b in zip(got, want))

    def native(*args):
        raise AssertionError("the function in C++ was called")
    monkeypatch.setattr(fa._native(), "attention", native)
    p, k, v = q.detach(), k.detach(), v.detach()
    with pytest.raises(AssertionError):
        fa.flash_attention(p, k, v)
    with pytest.raises(NotImplementedError), forward_ad.dual_level():
        fa.flash_attention(forward_ad.make_dual(p, p), k, v)
    for transformed in (lambda: torch.func.jvp(lambda x: fa.flash_attention(x, k, v), (p,), (p,)), lambda: torch.func.vjp(lambda x: fa.flash_attention(x, k, v), p),
                        lambda: torch.func.vmap(lambda x: fa.flash_attention(x, k, v))(torch.stack([p, p]))):
        with pytest.raises(RuntimeError, match="functorch"):
            transformed()
    traced = torch.jit.trace(lambda x: fa.flash_attention(x, k, v), (p,), check_trace=False)
    assert traced(p).shape == p.shape
    assert torch.equal(_python(torch, fa, p, k, v), want[0])


def test_other_streams_and_threads(fa):
    import threading
    import torch
    q, k, v, do = _inputs(torch, 6, 256, 64, 4, 4, False, torch.float16)
    o = fa.flash_attention(q, k, v, causal=True)
    want = (o.detach(),) + torch.autograd.grad(o, (q, k, v), do)
    torch.cuda.synchronize()
    failed = []

    def work():
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            for _ in range(20):
                x = fa.flash_attention(q, k, v, causal=True)
                got = (x.detach(),) + torch.autograd.grad(x, (q, k, v), do)
                stream.synchronize()
                if not all(torch.equal(a, b) for a, b in zip(got, want)):
                    failed.append(1)
    threads = [threading.Thread(target=work) for _ in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed
