"""The work that programs have this framework do, as cases for timing.

A case is one feed-forward step of a decoder layer through :class:`fairseq2_amd.MoE`: generation steps of a
few sequences, prompts and chunks of prompts, and training steps, over the layer sizes, number formats and
routing conventions of this repository's workloads, its tests and its notes.

Fields of a case: ``tokens`` rows of ``dim`` features go through ``top_k`` of ``experts`` SwiGLU networks of
``inner`` features (and one shared network where ``shared``).  ``act`` is the type of rows and parameters,
``weights`` the format of the expert weights (``"e4m3"``: quantised once when they are loaded), ``mx`` the
option that quantises the rows as well.  ``mode`` is ``"reference"`` (sigmoid, rows scaled on the way in) or
``"softmax"`` (renormalised, results weighted).  ``skew`` is the exponent of the experts' popularity law (0: what
random rows give).  ``step`` is ``"layer"`` or ``"prenorm"`` (``x + layer(rms_norm(x))`` in one call), ``pass`` is
``"forward"``, ``"graph"`` (the same, recorded once into a HIP graph and replayed) or ``"train"`` (forward and
backward, every gradient).
"""

import math

import numpy as np
import torch

from fairseq2_amd import GraphedForward, MoE

_DTYPE = {"fp32": torch.float32, "bf16": torch.bfloat16}


def _case(tokens, dim, inner, experts, top_k, **more):
    case = {"tokens": tokens, "dim": dim, "inner": inner, "experts": experts, "top_k": top_k, "act": "bf16",
            "weights": "same", "mx": False, "shared": False, "mode": "softmax", "skew": 0.0, "step": "layer",
            "pass": "forward"}
    unknown = set(more) - set(case) - {"name"}
    if unknown:
        raise ValueError(f"no such fields: {sorted(unknown)}")
    return {**case, **more}


def listed():
    return [
        # One sequence generating: the latency of a step that reads eight experts and launches five kernels.
        _case(1, 2048, 768, 128, 8, skew=1.2, step="prenorm", name="decode_1"),
        # A small batch generating under a recorded graph, as serving loops run it.
        _case(8, 2048, 768, 128, 8, skew=1.2, step="prenorm", **{"pass": "graph"}, name="decode_8_graph"),
        # Large experts with a shared one, in the reference's routing mode, for a handful of sequences.
        _case(5, 5120, 8192, 16, 1, shared=True, mode="reference", name="decode_5_shared"),
        # A busy server's batch of sequences, weights as trained.
        _case(48, 2048, 768, 128, 8, skew=1.2, step="prenorm", name="decode_48"),
        # The same kind of batch with the experts stored in one byte.
        _case(64, 2048, 768, 128, 8, weights="e4m3", skew=1.2, name="decode_64_e4m3"),
        # A short prompt, or one chunk of a long one: a ragged number of rows over 64 experts.
        _case(777, 2048, 1024, 64, 8, step="prenorm", name="chunk_777"),
        # Prompts of a batch, many small experts with a skewed load (the default benchmark's layer).
        _case(8192, 2048, 768, 128, 8, skew=1.2, name="prefill_8192"),
        # Prompts of a batch, few large experts: the largest forward pass.
        _case(8192, 4096, 14336, 8, 2, skew=1.1, name="prefill_large"),
        # Prompts on the fp8 matrix pipe.
        _case(5000, 2048, 768, 128, 8, weights="e4m3", mx=True, skew=1.2, step="prenorm", name="prefill_5000_mx"),
        # A training step over many small experts.
        _case(4096, 2048, 768, 128, 8, step="prenorm", **{"pass": "train"}, name="train_4096"),
        # A training step with a shared expert in the reference's mode, the inner size as the reference's
        # constructor derives it (4096 * 2/3, halved, up to a multiple of 8), an odd number of rows.
        _case(3001, 1024, 1368, 16, 2, shared=True, mode="reference", **{"pass": "train"}, name="train_3001_shared"),
        # Fine-tuning or debugging in full precision.
        _case(1000, 512, 1408, 8, 2, act="fp32", mode="reference", **{"pass": "train"}, name="train_1000_fp32"),
    ]


def _log(rng, low, high):
    return math.exp(rng.uniform(math.log(low), math.log(high)))


def _layer_sizes(rng, step):
    """Sizes of a layer: many small experts, or few large ones; ``step`` is what ``inner`` is a multiple of."""
    if rng.random() < 0.5:
        experts, low, high, ks = rng.choice((32, 60, 64, 128)), 512, 2048, (4, 6, 8)
    else:
        experts, low, high, ks = rng.choice((8, 16)), 1024, 14336, (1, 2)
    dim = 64 * round(_log(rng, 512, 5120) / 64)
    inner = step * round(_log(rng, low, high) / step)
    return dim, inner, experts, rng.choice(ks)


def _draw(rng):
    kind = rng.choice(("decode", "decode", "decode_e4m3", "chunk", "prefill", "prefill_e4m3", "train", "train", "fp32"))
    more = {"mode": rng.choice(("softmax", "softmax", "reference")), "skew": rng.choice((0.0, 1.1, 1.2)),
            "step": rng.choice(("layer", "prenorm"))}
    if kind.endswith("_e4m3"):
        more.update(weights="e4m3", mx=kind.startswith("prefill") and rng.random() < 0.5, mode="softmax")
    else:
        more["shared"] = rng.random() < 0.3
    step = 64 if kind.endswith("_e4m3") else rng.choice((8, 64, 64))
    if kind.startswith("decode"):
        tokens = round(_log(rng, 1, 256))
        more["pass"] = rng.choice(("forward", "forward", "graph"))
    elif kind == "chunk":
        tokens = round(_log(rng, 257, 2048))
    elif kind.startswith("prefill"):
        tokens = round(_log(rng, 1025, 16384))
    elif kind == "train":
        tokens = round(_log(rng, 256, 8192))
        more["pass"] = "train"
    else:
        tokens = round(_log(rng, 64, 4096))
        more.update({"act": "fp32", "pass": rng.choice(("forward", "train"))})
    dim, inner, experts, top_k = _layer_sizes(rng, 128 if more.get("mx") else step)
    if more.get("mx"):
        dim = 128 * round(dim / 128)
    if kind == "fp32":  # models of a size that is trained or checked in full precision
        dim, inner = min(dim, 1024), min(inner, 2048)
    return _case(tokens, dim, inner, experts, top_k, **more)


def draw(rng):
    top = max((work(c) for c in listed()), key=lambda w: w["flops"])
    while True:
        case = _draw(rng)
        w = work(case)
        # (fp32 products run at a sixteenth of the bf16 rate)
        if w["flops"] * (16 if case["act"] == "fp32" else 1) <= top["flops"] and w["bytes"] <= 2 * top["bytes"]:
            return case


def _popularity(case):
    """What a popularity law adds to the logits of the experts in order of rank."""
    return -case["skew"] * np.log(np.arange(case["experts"]) + 1.0)


def _module(case, generator):
    prev = torch.get_default_dtype()
    torch.set_default_dtype(_DTYPE[case["act"]])
    try:
        with torch.device("cuda"):
            layer = MoE(
                case["dim"], case["inner"], case["shared"], case["experts"], 1.0, case["top_k"],
                inner_dim_scale=1.0, auto_scale=False,
                score_fn="sigmoid" if case["mode"] == "reference" else "softmax",
                renormalize=case["mode"] != "reference",
                scale_on="input" if case["mode"] == "reference" else "output",
                router_bias=case["skew"] > 0, act_quant="mxfp8" if case["mx"] else None,
            )
            norm = torch.nn.RMSNorm(case["dim"], eps=1e-6) if case["step"] == "prenorm" else None
    finally:
        torch.set_default_dtype(prev)
    with torch.no_grad():
        for p in layer.parameters():
            p.normal_(0.0, 0.02, generator=generator)
        if norm is not None:
            norm.weight.normal_(1.0, 0.1, generator=generator)
        if case["skew"] > 0:
            bias = torch.from_numpy(_popularity(case)).to(layer.router_bias)
            layer.router_bias.copy_(bias[torch.randperm(case["experts"], generator=generator, device="cuda")])
        if case["weights"] == "e4m3":
            layer.experts.quantize_fp8_()
    train = case["pass"] == "train"
    layer.requires_grad_(train).train(train)
    if norm is not None:
        norm.requires_grad_(train)
    return layer, norm


def prepare(case, seed):
    g = torch.Generator("cuda").manual_seed(seed)
    layer, norm = _module(case, g)
    dtype = _DTYPE[case["act"]]
    shape = (1, case["tokens"], case["dim"])
    x = torch.randn(shape, generator=g, device="cuda").to(dtype)
    state = {"pass": case["pass"], "layer": layer, "norm": norm, "x": x}
    if case["pass"] == "train":
        x.requires_grad_(True)
        # what the rest of the model sends back
        state["dout"] = torch.randn(shape, generator=g, device="cuda").to(dtype)
        params = {"x": x, **dict(layer.named_parameters())}
        if norm is not None:
            params["norm.weight"] = norm.weight
        state["params"] = params
    elif case["pass"] == "graph":
        state["graph"] = GraphedForward(layer, x, add_input=norm is not None, norm=norm)
    return state


def _call(state):
    x, norm = state["x"], state["norm"]
    return state["layer"](x) if norm is None else state["layer"](x, residual=x, norm=norm)


def run(state):
    if state["pass"] == "train":
        out = _call(state)
        names = list(state["params"])
        grads = torch.autograd.grad(out, [state["params"][n] for n in names], state["dout"])
        return {"out": out, **dict(zip(names, grads))}
    if state["pass"] == "graph":
        return state["graph"](state["x"])
    with torch.inference_mode():
        return _call(state)


def _active_experts(case):
    """How many experts the rows reach, from rows like those of :func:`prepare`."""
    tokens, experts = min(case["tokens"], 512), case["experts"]
    rng = np.random.default_rng(0)
    logits = 0.02 * math.sqrt(case["dim"]) * rng.standard_normal((tokens, experts))
    if case["skew"] > 0:
        logits += _popularity(case)
    return len(np.unique(np.argsort(-logits, axis=1)[:, : case["top_k"]]))


def work(case):
    tokens, dim, inner = case["tokens"], case["dim"], case["inner"]
    size = 4 if case["act"] == "fp32" else 2
    networks = case["top_k"] + int(case["shared"])
    flops = tokens * (6 * networks * dim * inner + 2 * dim * case["experts"])
    rows = tokens * dim * size  # of each of x, out and, in training, the two gradients
    router = dim * case["experts"] * size
    shared = 3 * dim * inner * size * int(case["shared"])
    expert = 3 * dim * inner * (1 if case["weights"] == "e4m3" else size)
    read = _active_experts(case) * expert + shared + router
    if case["pass"] != "train":
        return {"bytes": 2 * rows + read, "flops": flops}
    # every parameter has a gradient, of experts without rows too
    written = case["experts"] * expert + shared + router
    return {"bytes": 4 * rows + read + written, "flops": 3 * flops}


def tolerance(case):
    # rows, intermediates and results are rounded to 8 bits between f32 sums; in fp32 only the sums' order is free
    return {"rel": 1e-5 if case["act"] == "fp32" else 1e-2}
