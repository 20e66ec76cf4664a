"""Timed cases: the work a program built on this package has it do.

Each case is one call (or one forward with its backward) of a public entry point, at sizes from this
repository's configurations, models, tests and benchmark, or generic ones of the same kind.  ``kind`` says
what is called:

``train``   an attention layer inside a training step: forward, then the gradients of q, k and v
``infer``   attention without gradients (evaluation of a classifier, scoring of a text)
``prompt``  the first block of tokens of a generation on the moment state: its outputs and the new state
``step``    one further token on that state
``cached``  new tokens against cached keys and values (causal, the queries are the last tokens)

``front`` is how a program reaches the kernels: ``function`` the autograd function with the reference's
argument list, ``model`` the helper the transformer blocks call (the max-norm scaling of q and k with its
gradient), ``score`` the score-function front (q and k centred over tokens and scaled).  ``layout`` is where q,
k and v come from: ``heads`` contiguous (b, h, n, d), ``proj`` the transposed views of (b, n, h*d) projections.
"""
import math

import torch

from reproducing_fastmax_results_amd.attention_mechanisms.score_function import (
    FASTMultiHeadAttention_Function, FastmaxDecodeState, fastmax)
from reproducing_fastmax_results_amd.transformer.model import fastmax_attention


def _case(kind, b, h, n, d, dtype, mask=True, p=2, front="function", layout="heads", nk=None, scale=1.0, **name):
    return dict(kind=kind, front=front, b=b, h=h, n=n, nk=n if nk is None else nk, d=d, dtype=dtype, mask=mask, p=p,
                layout=layout, scale=scale, **name)


def listed():
    return [
        # The smallest ordinary call: unmasked fp32 attention of two heads of 32, where launches and the host's
        # part are the whole time (the shape the CPU algorithm is run on as well).
        _case("infer", 1, 2, 256, 32, "f32", mask=False, name="small_infer_f32"),
        # A layer of the image classifier: 256 images of 49 patches and a class token, 4 heads of 32, fp32, q and k
        # max-normalised.  Many short, odd sequences.
        _case("train", 256, 4, 50, 32, "f32", mask=False, front="model", layout="proj", name="classifier_train_f32"),
        # A layer of the decoder-only language model: 16 sequences of 1024 tokens, 8 heads of 64, bf16, normalised.
        _case("train", 16, 8, 1024, 64, "bf16", front="model", layout="proj", name="decoder_train_bf16"),
        # The benchmark's shape, in both types.
        _case("train", 4, 8, 4096, 64, "bf16", name="headline_train_bf16"),
        _case("train", 4, 8, 4096, 64, "f32", name="headline_train_f32"),
        # The score-function front on a ragged fp32 problem with a head size the kernels pad.
        _case("train", 3, 5, 777, 48, "f32", front="score", name="ragged_score_train_f32"),
        # Long contexts, order 2 and order 1.
        _case("train", 1, 16, 65536, 64, "bf16", p=2, scale=0.5, name="long_order2_train_bf16"),
        _case("train", 1, 16, 65536, 64, "bf16", p=1, scale=0.5, name="long_order1_train_bf16"),
        # Heads of 128.
        _case("train", 2, 8, 2048, 128, "bf16", layout="proj", name="wide_head_train_bf16"),
        # Generation: the prompt of one user (odd length), a token on the moment state, a token on cached keys.
        _case("prompt", 1, 16, 3001, 64, "bf16", layout="proj", name="prompt_bf16"),
        _case("step", 1, 16, 1, 64, "bf16", layout="proj", nk=1024, name="state_step_bf16"),
        _case("cached", 4, 8, 1, 64, "bf16", layout="proj", nk=4097, name="cached_step_bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# products of b*h*n*n (dense) and tokens b*h*n that a drawn training case may not exceed, per type
_MAX_PAIRS, _MAX_TOKENS = 32 * 4096 * 4096, 16 * 65536


def draw(rng):
    kind = rng.choice(["infer", "train", "train", "train", "train", "prompt", "step", "cached"])
    dtype = rng.choice(["f32", "bf16", "bf16"])
    layout = rng.choice(["heads", "proj"])
    if kind == "train":
        size = rng.choice(["many_short", "ordinary", "long", "wide"])
        if size == "many_short":
            return _case("train", _log(rng, 16, 256), rng.choice([4, 8]), _log(rng, 33, 256), rng.choice([32, 64]), dtype,
                         mask=rng.random() < 0.5, p=rng.choice([1, 2]), front=rng.choice(["model", "function"]), layout=layout)
        if size == "ordinary":
            n = _log(rng, 256, 4096)
            h = rng.choice([4, 8, 12])
            b = max(1, min(_log(rng, 1, 16), _MAX_PAIRS // (h * n * n)))
            front = rng.choice(["model", "function", "score"])
            return _case("train", b, h, n, rng.choice([32, 48, 64]), dtype, mask=rng.random() < 0.75,
                         p=rng.choice([1, 2, 2]), front=front, layout=layout)
        if size == "long":
            n = _log(rng, 8192, 65536)
            h = max(1, min(16, _MAX_TOKENS // n))
            return _case("train", 1, h, n, 64, "bf16", p=rng.choice([1, 2]), layout=layout, scale=0.5)
        return _case("train", rng.choice([1, 2]), 8, _log(rng, 256, 2048), rng.choice([96, 128]), "bf16",
                     mask=rng.random() < 0.75, layout=layout)
    if kind == "infer":
        return _case("infer", rng.choice([1, 2, 4]), rng.choice([2, 4, 8]), _log(rng, 64, 4096), rng.choice([32, 64]), dtype,
                     mask=rng.random() < 0.5, p=rng.choice([1, 2]), front=rng.choice(["model", "function"]), layout=layout)
    b, h = rng.choice([1, 2, 4]), rng.choice([8, 16])
    if kind == "prompt":
        return _case("prompt", b, h, _log(rng, 64, 4096), 64, dtype, p=rng.choice([1, 2, 2]), layout=layout)
    if kind == "step":
        return _case("step", b, h, 1, rng.choice([32, 64]), dtype, p=rng.choice([1, 2, 2]), layout=layout, nk=_log(rng, 64, 2048))
    n = rng.choice([1, 1, 1, _log(rng, 2, 64)])
    return _case("cached", b, h, n, rng.choice([32, 64]), dtype, p=rng.choice([1, 2, 2]), layout=layout, nk=n + _log(rng, 256, 16384))


def _dtype(case):
    return torch.bfloat16 if case["dtype"] == "bf16" else torch.float32


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    b, h, d = case["b"], case["h"], case["d"]

    def rows(n):
        if case["layout"] == "proj":
            x = torch.randn(b, n, h, d, generator=gen, device="cuda").transpose(1, 2)
        else:
            x = torch.randn(b, h, n, d, generator=gen, device="cuda")
        return (x * case["scale"]).to(_dtype(case))

    tau = 1.0 if case["front"] == "model" else 8.0 * math.sqrt(d)
    state = dict(case=case, tau=tau, q=rows(case["n"]))
    if case["kind"] == "step":
        # the state after a prompt of nk tokens, and one new token
        state["decode"] = FastmaxDecodeState(temperature=tau, p=case["p"])
        state["decode"].prompt(rows(case["nk"]), rows(case["nk"]), rows(case["nk"]))
        state["k"], state["v"] = rows(1), rows(1)
        return state
    state["k"], state["v"] = rows(case["nk"]), rows(case["nk"])
    if case["kind"] == "train":
        state["go"] = rows(case["n"])
        for name in ("q", "k", "v"):
            state[name] = state[name].detach().requires_grad_(True)
    return state


def _attention(case, q, k, v, tau):
    if case["front"] == "model":
        return fastmax_attention(q, k, v, mask=case["mask"], normalize=True, lim=1.0, temperature=tau, a0=1.0, a1=1.0, a2=0.5,
                                 p=case["p"])
    if case["front"] == "score":
        return fastmax(q, k, v, mask=case["mask"], normalize=1, p=case["p"])
    return FASTMultiHeadAttention_Function.apply(q, k, v, None, None, case["mask"], 0.0, False, tau, 1.0, 1.0, 0.5, 1.0, case["p"])


def run(state):
    case, q, k, v = state["case"], state["q"], state["k"], state["v"]
    kind = case["kind"]
    if kind == "step":
        return {"o": state["decode"].step(q, k, v), "state": state["decode"].state}
    if kind == "prompt":
        st = FastmaxDecodeState(temperature=state["tau"], p=case["p"])
        o = st.prompt(q, k, v)
        return {"o": o, "state": st.state}
    if kind == "train":
        o = _attention(case, q, k, v, state["tau"])
        dq, dk, dv = torch.autograd.grad(o, (q, k, v), state["go"])
        return {"o": o.detach(), "dq": dq, "dk": dk, "dv": dv}
    with torch.no_grad():
        return {"o": _attention(case, q, k, v, state["tau"])}


def work(case):
    """Bytes: inputs read once, outputs written once.  Operations: the cheaper of the two forms the result has,
    products with every visible key, or sums over key moments (the symmetric order-2 part counted once)."""
    bh, n, nk, d = case["b"] * case["h"], case["n"], case["nk"], case["d"]
    e = 2 if case["dtype"] == "bf16" else 4
    moments = d + (d * (d + 1) // 2 if case["p"] == 2 else 0)
    row = bh * d * e
    if case["kind"] == "step":
        state = 4 * bh * (1 + moments) * (d + 1)
        return {"bytes": 2 * state + 4 * row, "flops": 4 * bh * moments * (d + 1)}
    causal = case["mask"] or case["kind"] in ("prompt", "cached")
    keys = nk - (n - 1) / 2 if causal else nk                  # visible keys, the average over the queries
    dense = 2 * d * n * keys                                   # one product of all visible pairs
    unit = 2 * moments * (d + 1)                               # one token into, or out of, the moments
    if case["kind"] == "train":
        # forward 2 products, backward 5; or key and query moments summed, outputs and three gradients read out of them
        return {"bytes": 4 * (n + nk) * row, "flops": bh * min(7 * dense, 3 * unit * (n + nk))}
    flops = bh * min(2 * dense, unit * (n + nk))
    io = (2 * n + 2 * nk) * row
    if case["kind"] == "prompt":
        return {"bytes": io + 4 * bh * (1 + moments) * (d + 1), "flops": flops + bh * unit * nk}
    return {"bytes": io, "flops": flops}


def tolerance(case):
    # bf16: results are rounded to 8 bits and computed from half-precision products (relative error 1.5e-3 to 3e-3
    # against 64-bit results).  fp32: 2e-7 to 5e-7 against 64-bit results.
    return {"rel": 8e-3} if case["dtype"] == "bf16" else {"rel": 2e-6}
