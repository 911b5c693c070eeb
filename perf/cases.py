"""The attention workloads whose time is tracked, through the package's public Python entry points.

Four kinds of call, the ones a user of this library makes:

* ``prefill``  flash_attention_forward on whole sequences (O and the logsumexp),
* ``decode``   flash_attention_forward of one or a few new queries per head against a key/value cache, key splits
               chosen by the library,
* ``chunk``    the same for a chunk of a prompt behind the part of it that is already in the cache,
* ``train``    flash_attention under autograd: O, and dQ, dK, dV from a given dO.

``listed`` holds fixed sizes (the benchmark's configurations c1-c5, d1, d2 and generic ones), ``draw`` gives others
of the same ranges.
"""
import importlib.util
import math
import os
import sys

import torch


def _package():
    """The package of the working folder (its directory name has a hyphen, so it is loaded by path)."""
    name = "flash_attn_rtx5060_amd"
    if name not in sys.modules:
        path = os.path.join(os.getcwd(), "flash-attn-rtx5060_amd", "__init__.py")
        spec = importlib.util.spec_from_file_location(name, path)
        module = importlib.util.module_from_spec(spec)
        sys.modules[name] = module
        spec.loader.exec_module(module)
    return sys.modules[name]


def _case(kind, dtype, B, H, Hk, S, Sk, D, causal=True, window=-1, bshd=False, alibi=False, dropout=0.0, sigma=1.0,
          outliers=0.0, name=None):
    """Hk K/V heads under H query heads, S queries behind Sk keys (the queries are the last S positions), window: keys
    visible to the left (-1 all), bshd: stored [B, S, H, D] instead of [B, H, S, D], sigma: standard deviation of Q, K,
    V, outliers: share of the rows of Q that are eight times as large."""
    c = dict(kind=kind, dtype=dtype, B=B, H=H, Hk=Hk, S=S, Sk=Sk, D=D, causal=causal, window=window, bshd=bshd,
             alibi=alibi, dropout=dropout, sigma=sigma, outliers=outliers)
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # c1: a few heads of one short sequence; the smallest call, launch and host time
        _case("prefill", "fp16", 1, 4, 4, 256, 256, 64, causal=False, name="prefill_tiny"),
        # c2: a batch of ordinary sequences, head dimension 64
        _case("prefill", "fp16", 4, 16, 16, 2048, 2048, 64, name="prefill_d64"),
        # c3, the headline shape: long causal sequences, head dimension 128
        _case("prefill", "fp16", 2, 32, 32, 8192, 8192, 128, name="prefill_headline"),
        # c4: sliding-window layers of a long-context model
        _case("prefill", "bf16", 1, 32, 32, 16384, 16384, 128, window=1024, name="prefill_window"),
        # c5: one very long document; a hundredth of the queries is large, as real activations have it
        _case("prefill", "fp16", 1, 64, 64, 32768, 32768, 128, sigma=0.5, outliers=0.01, name="prefill_long"),
        # one user's next token behind a short, ragged cache: latency
        _case("decode", "bf16", 1, 32, 8, 1, 1003, 128, bshd=True, name="decode_single"),
        # d1: a serving batch with grouped K/V heads
        _case("decode", "fp16", 16, 32, 8, 1, 8192, 128, name="decode_batch"),
        # d2: long caches, one K/V head per query head
        _case("decode", "fp16", 4, 32, 32, 1, 32768, 128, name="decode_long"),
        # a chunk of a prompt behind what is already cached (ragged, [B, S, H, D] as a projection leaves it)
        _case("chunk", "bf16", 1, 32, 8, 500, 4596, 128, bshd=True, name="chunk_prefill"),
        # a training step of a decoder with grouped K/V heads, stored [B, S, H, D]
        _case("train", "bf16", 2, 32, 8, 4096, 4096, 128, bshd=True, name="train_gqa"),
        # a training step on sequences of no round length, head dimension 64
        _case("train", "fp16", 8, 16, 16, 1000, 1000, 64, name="train_ragged"),
        # an encoder's training step: short sequences, no mask, dropout
        _case("train", "fp16", 16, 16, 16, 512, 512, 64, causal=False, bshd=True, dropout=0.1, name="train_dropout"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _length(rng, lo, hi):
    """Half of the lengths a multiple of 128, the others as they come."""
    n = _log(rng, lo, hi)
    return max(128, n // 128 * 128) if rng.random() < 0.5 else n


def draw(rng):
    while True:
        kind = rng.choice(("prefill", "prefill", "prefill", "decode", "decode", "chunk", "train", "train"))
        D = rng.choice((64, 128, 128))
        dtype = rng.choice(("fp16", "bf16"))
        H = rng.choice((4, 8, 16, 32, 32, 64))
        Hk = rng.choice((H, H, max(1, H // 4), max(1, H // 8)))
        bshd = rng.random() < 0.5
        if kind == "prefill":
            S = _length(rng, 128, 32768)
            c = _case(kind, dtype, _log(rng, 1, 32), H, Hk, S, S, D, causal=rng.random() < 0.75, bshd=bshd)
        elif kind == "decode":
            S = rng.choice((1, 1, 1, 2, 4))
            Sk = S + _log(rng, 100, 40000)
            c = _case(kind, dtype, _log(rng, 1, 64), H, Hk, S, Sk, D, bshd=bshd)
        elif kind == "chunk":
            S = _length(rng, 32, 2048)
            c = _case(kind, dtype, _log(rng, 1, 4), H, Hk, S, S + _log(rng, 256, 32768), D, bshd=bshd)
        else:
            S = _length(rng, 128, 16384)
            c = _case(kind, dtype, _log(rng, 1, 32), H, Hk, S, S, D, causal=rng.random() < 0.75, bshd=bshd)
        option = rng.random()
        if option < 0.15 and c["causal"] and c["Sk"] > 256:
            c["window"] = _log(rng, 128, c["Sk"] // 2)
        elif option < 0.25:
            c["alibi"] = True
        elif option < 0.35 and kind == "train":
            c["dropout"] = 0.1
        w = work(c)
        # from the smallest calls up to a tenth of the largest listed one, a few GB of cache at most
        if w["flops"] <= 1.8e12 and w["bytes"] <= 3e9:
            return c


def _pairs(c):
    """Visible (query, key) pairs per head."""
    S, Sk, w = c["S"], c["Sk"], c["window"]
    if not c["causal"]:
        return S * Sk
    total = 0
    for i in range(S):
        pos = i + Sk - S
        total += min(pos, w) + 1 if w >= 0 else pos + 1
    return total


def prepare(case, seed):
    c = case
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    dtype = torch.bfloat16 if c["dtype"] == "bf16" else torch.float16

    def tensor(heads, length, sigma, outliers=0.0):
        shape = (c["B"], length, heads, c["D"]) if c["bshd"] else (c["B"], heads, length, c["D"])
        t = torch.randn(shape, device="cuda", generator=gen)
        t *= sigma
        if outliers:
            t *= 1.0 + 7.0 * (torch.rand(shape[:3] + (1,), device="cuda", generator=gen) < outliers)
        t = t.to(dtype)
        return t.transpose(1, 2) if c["bshd"] else t

    q = tensor(c["H"], c["S"], c["sigma"], c["outliers"])
    k, v = tensor(c["Hk"], c["Sk"], c["sigma"]), tensor(c["Hk"], c["Sk"], c["sigma"])
    options = dict(causal=c["causal"], window_left=c["window"])
    if c["alibi"]:
        # the usual geometric slopes
        options["alibi_slopes"] = torch.tensor([2.0 ** (-8.0 * (h + 1) / c["H"]) for h in range(c["H"])], device="cuda")
    if c["dropout"]:
        options.update(dropout_prob=c["dropout"], seed=48)
    state = dict(kind=c["kind"], q=q, k=k, v=v, options=options)
    if c["kind"] == "train":
        for t in (q, k, v):
            t.requires_grad_(True)
        state["do"] = tensor(c["H"], c["S"], 1.0)
    return state


def run(state):
    fa = _package()
    q, k, v, options = state["q"], state["k"], state["v"], state["options"]
    if state["kind"] == "prefill":
        return fa.flash_attention_forward(q, k, v, **options)
    if state["kind"] in ("decode", "chunk"):
        return fa.flash_attention_forward(q, k, v, splits="auto", return_lse=False, **options)
    o = fa.flash_attention(q, k, v, **options)
    return (o.detach(),) + torch.autograd.grad(o, (q, k, v), state["do"])


def work(case):
    c = case
    q, kv = 2.0 * c["B"] * c["H"] * c["S"] * c["D"], 2.0 * c["B"] * c["Hk"] * c["Sk"] * c["D"]
    product = 2.0 * c["B"] * c["H"] * c["D"] * _pairs(c)
    if c["kind"] == "train":
        # Q, K, V, dO in, O, dQ, dK, dV out; two products forward and five backward
        return {"bytes": 4.0 * q + 4.0 * kv, "flops": 7.0 * product}
    if c["kind"] != "prefill" and c["causal"] and c["window"] >= 0:
        # behind a window only the keys that some query sees
        kv *= min(1.0, (c["window"] + c["S"]) / c["Sk"])
    lse = 4.0 * c["B"] * c["H"] * c["S"] if c["kind"] == "prefill" else 0.0
    return {"bytes": 2.0 * q + 2.0 * kv + lse, "flops": 2.0 * product}


def tolerance(case):
    # Four times what these paths differ by from the same attention (and its gradients) in 64 bits on these inputs:
    # fp16 2.4e-4 to 3.3e-4, bf16 1.9e-3 to 2.7e-3 over O, dQ, dK and dV; single values up to 0.0105 and 0.068 of the
    # larger of the value and the root mean square (dQ and dK where a query sees a few keys only).
    return {"rel": 1e-2, "max": 0.28} if case["dtype"] == "bf16" else {"rel": 1.3e-3, "max": 0.042}
