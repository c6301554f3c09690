"""The work that programs built on e_natten_amd give it, as cases that can be timed.

A case is one call of a public entry point (``natten2d`` or ``natten1d``): a forward as in
inference, or a forward and backward as in one layer of a training step, through torch's autograd.
``listed()`` names one case for every use, ``draw()`` makes others of the same ranges.

Fields of a case
    op        "2d" or "1d"
    mode      "train" (forward and backward) or "infer" (forward of tensors without gradients)
    dtype     "bf16", "fp16" or "fp32"
    B, N      batch and heads
    H, W      image sides (2d); T: sequence length (1d)
    d, k      head_dim and kernel_size
    dilation, causal, rpb   the options of the same names (rpb: with a relative position bias)
    scaled    logits times head_dim ** -0.5, as a transformer layer has them, or unscaled as in the
              reference's own benchmark
    layout    "plain": q, k, v and the upstream gradient are contiguous [B, N, ..., d];
              "proj": q, k, v are the three views of one projection [B, ..., 3, N, d], and the
              upstream gradient a view of [B, ..., N, d], as a transformer layer has them
"""
import math

import torch

from e_natten_amd import natten1d, natten2d

_DTYPE = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_BASE = {"op": "2d", "mode": "train", "dtype": "bf16", "dilation": 1, "causal": False,
         "rpb": False, "scaled": True, "layout": "plain"}


def _case(**fields):
    return dict(_BASE, **fields)


def listed():
    return [
        # the smallest call: a float32 check-sized image, where only latency counts
        _case(name="check_fp32_16", dtype="fp32", B=1, N=2, H=16, W=16, d=32, k=3),
        # the reference's benchmark shape: forward alone, as an encoder at inference
        _case(name="readme_infer_256", mode="infer", scaled=False, B=4, N=4, H=256, W=256, d=128,
              k=5),
        # ... its forward and backward, the shape of the headline metric
        _case(name="readme_train_128", scaled=False, B=4, N=4, H=128, W=128, d=128, k=5),
        # ... and in float32, the type that the reference's benchmark runs in
        _case(name="readme_fp32_128", dtype="fp32", scaled=False, B=4, N=4, H=128, W=128, d=128,
              k=5),
        # a large window: overlapping neighborhoods, the most arithmetic per byte
        _case(name="window13_train", B=2, N=8, H=128, W=128, d=64, k=13),
        # vision backbone, first stage: large image, few narrow heads, views of one projection
        _case(name="backbone_stage1", layout="proj", B=8, N=2, H=112, W=112, d=32, k=7),
        # vision backbone, last stage: images of twice the window, launches and host time count
        _case(name="backbone_stage4", layout="proj", B=8, N=16, H=14, W=14, d=32, k=7),
        # vision backbone with a learned relative position bias, second stage
        _case(name="backbone_bias", layout="proj", rpb=True, B=8, N=4, H=56, W=56, d=32, k=7),
        # vision backbone with dilated neighborhoods, second stage
        _case(name="backbone_dilated", layout="proj", dilation=4, B=8, N=4, H=56, W=56, d=32, k=7),
        # odd sizes throughout: ragged image, head_dim between the powers of two, half precision
        _case(name="ragged_fp16", dtype="fp16", B=3, N=5, H=61, W=83, d=48, k=9),
        # sequence model with local windows, training
        _case(name="sequence_train", op="1d", B=4, N=8, T=16384, d=64, k=7),
        # sliding-window causal attention of a language model: reading a prompt
        _case(name="causal_prefill", op="1d", mode="infer", causal=True, layout="proj", B=1, N=16,
              T=8192, d=128, k=128),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# No drawn case moves more bytes or has more arithmetic than the largest listed ones.
_MAX_BYTES, _MAX_FLOPS = 1.4e9, 39e9


def _fit(case):
    """Halve the batch, then the heads, then the extents until the case is within the limits."""
    least = case["k"] * case["dilation"]
    while work(case)["bytes"] > _MAX_BYTES or work(case)["flops"] > _MAX_FLOPS:
        if case["B"] > 1:
            case["B"] //= 2
        elif case["N"] > 1:
            case["N"] //= 2
        elif case["op"] == "1d":
            case["T"] = max(least, case["T"] // 2)
        else:
            case["H"], case["W"] = max(least, case["H"] // 2), max(least, case["W"] // 2)
    return case


def draw(rng):
    """One more case: a use, then sizes over that use's whole range."""
    use = rng.choice(("image", "image", "image", "fp32", "backbone", "bias", "dilated", "sequence",
                      "sequence", "causal"))
    mode = rng.choice(("train", "train", "infer"))
    half = rng.choice(("bf16", "bf16", "fp16"))
    layout = rng.choice(("plain", "proj"))
    if use in ("sequence", "causal"):
        # the largest windows belong to causal models, whose kernel_size may be even
        k = _log_int(rng, 16, 512) if use == "causal" else 2 * _log_int(rng, 1, 48) + 1
        return _fit(_case(op="1d", mode=mode, dtype=half, layout=layout, causal=use == "causal",
                          B=rng.randint(1, 8), N=rng.randint(1, 16),
                          T=max(k, _log_int(rng, 100, 16384)),
                          d=rng.choice((32, 64, 64, 80, 128, 128)), k=k))
    B, N = rng.randint(1, 8), rng.randint(1, 16)
    H = _log_int(rng, 14, 256)
    W = H if rng.random() < 0.5 else max(14, min(256, int(H * rng.uniform(0.6, 1.6))))
    if use == "fp32":
        return _fit(_case(mode=mode, dtype="fp32", layout=layout, B=B, N=N, H=H, W=W,
                          d=rng.choice((32, 64, 128)), k=rng.choice((3, 5, 7))))
    if use == "image":
        return _fit(_case(mode=mode, dtype=half, layout=layout, scaled=rng.random() < 0.7, B=B, N=N,
                          H=H, W=W, d=rng.choice((32, 48, 64, 64, 96, 128, 128)),
                          k=rng.choice((3, 5, 7, 9, 11, 13) if min(H, W) > 13 else (3, 5, 7))))
    # vision backbones: narrow heads, small to middling windows, views of one projection
    k = rng.choice((5, 7, 7, 9))
    case = _case(mode=mode, dtype=half, layout="proj", rpb=use == "bias", B=B, N=N,
                 H=max(14, min(H, 128)), W=max(14, min(W, 128)), d=rng.choice((32, 32, 64)), k=k)
    if use == "dilated":
        case["dilation"] = dilation = rng.randint(2, 8)
        for side in ("H", "W"):
            case[side] = max(case[side], k * dilation)
    return _fit(case)


def _extent(case):
    return (case["T"],) if case["op"] == "1d" else (case["H"], case["W"])


def _tensor(gen, case, copies):
    """`copies` tensors [B, N, *extent, d] of N(0, 1) values in the case's layout."""
    B, N, d, ext = case["B"], case["N"], case["d"], _extent(case)
    dtype = _DTYPE[case["dtype"]]
    if case["layout"] == "plain":
        return [torch.randn((B, N, *ext, d), generator=gen, device="cuda", dtype=dtype)
                for _ in range(copies)]
    x = torch.randn((B, *ext, copies, N, d), generator=gen, device="cuda", dtype=dtype)
    at = len(ext) + 1
    return [t.movedim(at, 1) for t in x.unbind(at)]


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    train = case["mode"] == "train"
    qkv = [t.requires_grad_(train) for t in _tensor(gen, case, 3)]
    state = {"case": case, "qkv": qkv, "rpb": None,
             "options": {"scale": case["d"] ** -0.5 if case["scaled"] else 1.0,
                         "dilation": case["dilation"], "is_causal": case["causal"]}}
    if case["rpb"]:
        state["rpb"] = torch.randn((case["N"],) + (2 * case["k"] - 1,) * len(_extent(case)),
                                   generator=gen, device="cuda",
                                   dtype=_DTYPE[case["dtype"]]).requires_grad_(train)
    if train:
        state["grad"] = _tensor(gen, case, 1)[0]
    return state


def run(state):
    """One layer's attention: the output, and in training the gradients of q, k, v (and the bias)."""
    case, rpb = state["case"], state["rpb"]
    q, k, v = state["qkv"]
    natten = natten2d if case["op"] == "2d" else natten1d
    out = natten(q, k, v, case["k"], rpb=rpb, **state["options"])
    if case["mode"] == "infer":
        return out
    inputs = (q, k, v) if rpb is None else (q, k, v, rpb)
    return (out, *torch.autograd.grad(out, inputs, state["grad"]))


def work(case):
    """Bytes: the forward reads q, k, v and writes the output and a log-sum-exp per query; the
    backward, a call of its own whose upstream gradient depends on that output, reads q, k, v, the
    upstream gradient and the log-sum-exp and writes three gradients.  Operations: two products of
    length d per (query, key) pair forward, five backward."""
    ext = _extent(case)
    queries = case["B"] * case["N"] * math.prod(ext)
    tensor = queries * case["d"] * (4 if case["dtype"] == "fp32" else 2)
    if case["causal"]:  # the first queries of a sequence see fewer keys
        k, T = min(case["k"], case["T"]), case["T"]
        pairs = case["B"] * case["N"] * (k * T - k * (k - 1) // 2)
    else:
        pairs = queries * case["k"] ** len(ext)
    train = case["mode"] == "train"
    return {"bytes": (11 if train else 4) * tensor + (8 if train else 4) * queries,
            "flops": (14 if train else 4) * pairs * case["d"]}


def tolerance(case):
    """Four times what the present kernels differ by from the same path in float64, at reduced
    batch and sides: at most 2.9e-3 (bf16), 3.7e-4 (fp16) and 3.5e-7 (fp32); with unscaled logits
    of magnitude 50 the probabilities are sharper, and bf16 differs by 5.9e-3."""
    if case["dtype"] == "fp32":
        return {"rel": 2e-6}
    return {"rel": {"bf16": 1.2e-2, "fp16": 1.5e-3}[case["dtype"]] * (1 if case["scaled"] else 2)}
