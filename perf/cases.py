"""The calls whose speed counts: dynamic-mask attention as a model's training step, prefill and decode loop make it.

Three kinds of call, all through the package's public functions:

* "attention": `flash_sparse_attn_func` with a keep-mask (the `window` largest bias entries of a row) and a bias that the
  caller already holds.  `rows` says whether mask and bias have one row per query ("query") or one row that all queries
  share ("column"); `bias` can also be "none".
* "layer": what a dynamic-mask attention layer runs between its projections: `dynamic_mask_bias` over the value states,
  `create_mask` with an optional padding mask, then the attention.
* "ragged": `flash_sparse_attn_varlen_func` over sequences that lie back to back.

`train` adds the backward pass (gradients of everything that takes one); without it the call runs under no_grad, as
inference does.  Inputs are drawn from N(0, 1) as in the repository's benchmark, on the GPU, from the seed alone.
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "flash-dmattn_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from flash_sparse_attn import flash_sparse_attn_func, flash_sparse_attn_varlen_func  # noqa: E402
from flash_sparse_attn.utils.bias import dynamic_mask_bias  # noqa: E402
from flash_sparse_attn.utils.mask import create_mask  # noqa: E402

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def _attention(name, B, Lq, Lk, H, Hk, d, window, rows="column", bias="column", causal=True, train=False, dtype="bf16"):
    return {"name": name, "kind": "attention", "B": B, "Lq": Lq, "Lk": Lk, "H": H, "Hk": Hk, "d": d, "window": window,
            "rows": rows, "bias": bias, "causal": causal, "train": train, "dtype": dtype}


def _layer(name, B, Lq, Lk, H, Hk, d, window, padded=False, train=False, dtype="bf16"):
    return {"name": name, "kind": "layer", "B": B, "Lq": Lq, "Lk": Lk, "H": H, "Hk": Hk, "d": d, "window": window,
            "padded": padded, "train": train, "dtype": dtype}


def _ragged(name, lens, H, Hk, d, train=False, dtype="bf16"):
    return {"name": name, "kind": "ragged", "lens": ",".join(str(n) for n in lens), "H": H, "Hk": Hk, "d": d,
            "train": train, "dtype": dtype}


def listed():
    return [
        # the smallest training step (unit tests of a model, toy runs, the last short batch): launches and host work
        _attention("step_small", 1, 256, 256, 2, 1, 64, 128, train=True),
        # one token of one conversation, a cache whose length is whatever has been generated so far
        _attention("decode_one", 1, 1, 2049, 32, 8, 128, 512, causal=False),
        # a decode batch over long caches: bound by the kept K / V rows
        _attention("decode_long", 8, 1, 65536, 32, 8, 128, 2048, causal=False),
        # a whole layer of a decode step: bias of the cache's value states, top-k, attention; prompts padded on the left
        _layer("layer_decode", 8, 1, 4093, 32, 8, 128, 1024, padded=True),
        # prefill of a prompt, mask and bias in hand
        _attention("prefill_8k", 1, 8192, 8192, 32, 8, 128, 2048),
        # one chunk of a long prompt against the cache of the chunks before it
        _attention("prefill_chunk", 1, 512, 16384, 32, 8, 128, 2048),
        # a whole layer of a prefill: half precision, the widest head dimension, a ragged length
        _layer("layer_prefill_wide", 1, 3001, 3001, 8, 4, 256, 1024, dtype="fp16"),
        # a whole layer of a training step on short sequences, gradients on into the bias producer's parameters
        _layer("layer_train_2k", 4, 2048, 2048, 16, 8, 64, 512, train=True),
        # training on long sequences, a quarter of the keys kept
        _attention("train_8k", 1, 8192, 8192, 32, 8, 128, 2048, train=True),
        # a learned bias and a mask of its own for every query, with its gradient: bound by reading and writing them
        _attention("train_query_4k", 2, 4096, 4096, 16, 16, 64, 1024, rows="query", bias="query", train=True),
        # the same form at a ragged length, grouped heads that share mask and bias, the wider head, not causal
        _attention("train_query_odd", 1, 1999, 1999, 16, 4, 128, 512, rows="query", bias="query", causal=False, train=True, dtype="fp16"),
        # packed training sequences of very different lengths, no mask
        _ragged("ragged_train", [100, 3000, 777, 5000, 64, 2048, 1, 5394], 32, 8, 128, train=True),
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, even over the logarithm; half of them odd or otherwise not round."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    n = min(max(n, lo), hi)
    return n if rng.random() < 0.5 or n < 128 else n // 64 * 64


def _heads(rng):
    return rng.choice([(2, 1), (8, 2), (8, 4), (16, 4), (16, 8), (16, 16), (32, 8)])


def _draw_once(rng):
    what = rng.choice(["decode", "decode", "layer_decode", "prefill", "chunk", "layer_prefill", "layer_train", "train", "query", "ragged"])
    H, Hk = _heads(rng)
    d = rng.choice([64, 64, 96, 128, 128, 128, 256])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    if what in ("decode", "layer_decode"):
        B, Lk = _log(rng, 1, 16), _log(rng, 256, 65536 if what == "decode" else 16384)
        window = _log(rng, 128, 4096)
        if what == "decode":
            return _attention("", B, 1, Lk, H, Hk, d, min(window, Lk), causal=False, dtype=dtype)
        return _layer("", B, 1, Lk, H, Hk, d, min(window, Lk), padded=rng.random() < 0.5, dtype=dtype)
    if what == "ragged":
        lens = [_log(rng, 1, 6000) for _ in range(rng.randint(2, 12))]
        return _ragged("", lens, H, Hk, d, train=rng.random() < 0.5, dtype=dtype)
    B = rng.choice([1, 1, 2, 4])
    if what == "query":
        L = _log(rng, 128, 4096)
        return _attention("", B, L, L, H, Hk, d, min(_log(rng, 64, 2048), L), rows="query", bias=rng.choice(["query", "query", "column", "none"]),
                          causal=rng.random() < 0.7, train=rng.random() < 0.6, dtype=dtype)
    L = _log(rng, 64, 32768)
    window = min(_log(rng, 64, 4096), L)
    if what == "chunk":
        return _attention("", B, min(_log(rng, 16, 2048), L), L, H, Hk, d, window, dtype=dtype)
    if what in ("layer_prefill", "layer_train"):
        return _layer("", B, L, L, H, Hk, d, window, padded=rng.random() < 0.3, train=what == "layer_train", dtype=dtype)
    return _attention("", B, L, L, H, Hk, d, window, causal=rng.random() < 0.8, train=what == "train", dtype=dtype)


def _affordable(case):
    """No more than the largest listed case costs: the work of the calls is bounded, and with it what the wide head
    dimension, the dense ragged form and the per-query form (which reads the whole mask) may ask for."""
    w = work(case)
    flops = 4e11
    if case["d"] > 128:
        flops /= 4
    if case.get("rows") == "query" and case["B"] * case["H"] * case["Lq"] * case["Lk"] * case["d"] > 1.2e10:
        return False
    return w["flops"] <= flops and w["bytes"] <= 1.5e9


def draw(rng):
    while True:
        case = _draw_once(rng)
        case.pop("name")
        if _affordable(case):
            return case


def _normal(gen, dtype, *shape):
    return torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float32).to(dtype)


def _top(bias, window):
    """The keep-mask of the `window` largest entries of every row."""
    mask = torch.zeros(bias.shape, dtype=torch.bool, device=bias.device)
    for b in range(bias.shape[0]):  # (a slice at a time: the indices of a per-query mask take four times its bias)
        mask[b].scatter_(-1, bias[b].float().topk(window, dim=-1, sorted=False).indices, True)
    return mask


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype, train = _DTYPES[case["dtype"]], case["train"]
    H, Hk, d = case["H"], case["Hk"], case["d"]
    s = {"case": case, "wanted": []}

    def leaf(t):
        if train:
            t.requires_grad_(True)
            s["wanted"].append(t)
        return t

    if case["kind"] == "ragged":
        lens = [int(n) for n in case["lens"].split(",")]
        total = sum(lens)
        s["q"] = leaf(_normal(gen, dtype, total, H, d))
        s["k"] = leaf(_normal(gen, dtype, total, Hk, d))
        s["v"] = leaf(_normal(gen, dtype, total, Hk, d))
        first = [0]
        for n in lens:
            first.append(first[-1] + n)
        s["cu"] = torch.tensor(first, dtype=torch.int32, device="cuda")
        s["longest"] = max(lens)
        if train:
            s["dout"] = _normal(gen, dtype, total, H, d)
        return s

    B, Lq, Lk = case["B"], case["Lq"], case["Lk"]
    s["q"] = leaf(_normal(gen, dtype, B, Lq, H, d))
    s["k"] = leaf(_normal(gen, dtype, B, Lk, Hk, d))
    s["v"] = leaf(_normal(gen, dtype, B, Lk, Hk, d))
    if train:
        s["dout"] = _normal(gen, dtype, B, Lq, H, d)
    if case["kind"] == "layer":
        s["w"] = leaf((torch.randn(Hk, Hk * d, generator=gen, device="cuda") * 0.5 / math.sqrt(Hk * d)).to(dtype))
        s["a"] = leaf(torch.linspace(0.5, 1.5, Hk, device="cuda").to(dtype))
        s["padding"] = None
        if case["padded"]:  # prompts of different lengths, padded on the left
            pads = torch.randint(0, Lk // 4 + 1, (B, 1), generator=gen, device="cuda")
            s["padding"] = torch.arange(Lk, device="cuda")[None, :] >= pads
        return s
    query = case["rows"] == "query"
    scores = _normal(gen, dtype, B, Hk, Lq if query else 1, Lk)
    s["mask"] = _top(scores, case["window"])
    if case["bias"] == "none":
        s["bias"] = None
    elif case["bias"] == case["rows"]:
        s["bias"] = leaf(scores)
    else:
        s["bias"] = leaf(_normal(gen, dtype, B, Hk, 1, Lk))
    return s


def _forward(s):
    case = s["case"]
    if case["kind"] == "ragged":
        n = s["longest"]
        return flash_sparse_attn_varlen_func(s["q"], s["k"], s["v"], s["cu"], s["cu"], n, n, is_causal=True)
    if case["kind"] == "layer":
        bias = dynamic_mask_bias(s["v"], s["w"], s["a"])
        mask = create_mask(bias, s["padding"], case["B"], case["Lq"], case["Lk"], case["window"],
                           torch.finfo(bias.dtype).min, type="topk")
        return flash_sparse_attn_func(s["q"], s["k"], s["v"], mask, bias, is_causal=case["Lq"] > 1)
    return flash_sparse_attn_func(s["q"], s["k"], s["v"], s["mask"], s["bias"], is_causal=case["causal"])


def run(s):
    if not s["case"]["train"]:
        with torch.no_grad():
            return _forward(s)
    out = _forward(s)
    return (out.detach(),) + torch.autograd.grad(out, s["wanted"], s["dout"])


def work(case):
    H, Hk, d, train = case["H"], case["Hk"], case["d"], case["train"]
    e = 2  # bytes of an element
    if case["kind"] == "ragged":
        lens = [int(n) for n in case["lens"].split(",")]
        pairs = H * sum(n * (n + 1) // 2 for n in lens)
        rows = sum(lens)
        size = e * d * rows * ((H * 2 + Hk * 2) + (H * 2 + Hk * 2 if train else 0))
        return {"bytes": size, "flops": (14 if train else 4) * d * pairs}
    B, Lq, Lk = case["B"], case["Lq"], case["Lk"]
    kept = min(case["window"], Lk)
    causal = Lq > 1 and case.get("causal", True)
    visible = [max(0, min(Lk, i + 1 + Lk - Lq)) for i in (0, Lq - 1)]
    if not causal:
        scores = Lq * Lk
    elif Lq <= Lk:
        scores = Lq * (visible[0] + visible[1]) // 2
    else:
        scores = Lk * (Lk + 1) // 2
    pairs = B * H * scores * kept // Lk  # (the kept keys lie evenly over the row)
    flops = (14 if train else 4) * d * pairs
    size = e * d * B * Lq * H * (4 if train else 2)  # q, out (dout, dq)
    if case["kind"] == "layer":
        flops += (6 if train else 2) * Hk * Hk * d * B * Lk
        size += e * d * B * Hk * (kept + Lk) + (e * d * B * Hk * 2 * Lk if train else 0)  # kept K, all of V; dK, dV
        size += B * Lk if case["padded"] else 0
        return {"bytes": size, "flops": flops}
    if case["rows"] == "column":
        size += 2 * e * d * B * Hk * kept + B * Hk * (Lk + e * kept)  # kept K and V rows, the mask, the kept keys' bias
        size += (2 * e * d * B * Hk * Lk + e * B * Hk * Lk if train else 0)  # dK, dV, dBias
        return {"bytes": size, "flops": flops}
    size += 2 * e * d * B * Hk * Lk * (2 if train else 1) + B * Hk * scores  # K, V (dK, dV), the visible part of the mask
    if case["bias"] != "none":
        bias = (scores, Lq * Lk) if case["bias"] == "query" else (Lk, Lk)
        size += e * B * Hk * (bias[0] + (bias[1] if train else 0))
    return {"bytes": size, "flops": flops}


def tolerance(case):
    """Probabilities and dS are rounded to the inputs' 16-bit type before the second contractions, and so are the
    results: half a unit in the last place is 2^-9 (bf16) or 2^-12 (fp16) of a value, and a few such roundings meet."""
    return {"rel": 1e-2} if case["dtype"] == "bf16" else {"rel": 2.5e-3}
