"""The work a user of the fused normalisations has them do, as cases that can be timed and compared.

A case is one call site of a transformer block, at one size: the modulated LayerNorm of a block's entry, the
gated residual update with the norm behind it, the per-head RMSNorm of queries and keys (from the fused
projection, with or without the rotary embedding, or on the transposed view the plain attention module passes)
and RMSNorm over the hidden dimension.  `train` cases run forward and backward through autograd and return the
outputs and every gradient; the others run the forward pass alone, as inference and the first pass of
activation recompute do.  Sequence lengths are those of a 129-frame 720p clip (118 800 image tokens, 29 700 on one
of four context-parallel ranks), of shorter clips and of the text stream (at most 256 tokens).
"""
import os

import torch

# The switch a training script exports: the module forms take the fused path.
os.environ.setdefault("FUSED_KERNELS", "1")

from teletron_amd import fusedlayers as FL  # noqa: E402

EPS = 1e-6
_TYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_ELEM = {"bf16": 2, "fp16": 2, "fp32": 4}

# Bytes of tensors the largest listed case moves; a drawn case stays below it.
_LARGEST = 5 * 118800 * 3072 * 2


def _norm(name, kind, batch, tokens, hidden, dtype, train):
    return {"name": name, "kind": kind, "batch": batch, "tokens": tokens, "hidden": hidden, "dtype": dtype, "train": train}


def _heads(name, kind, batch, tokens, heads, head_dim, rotated, dtype, train):
    return {"name": name, "kind": kind, "batch": batch, "tokens": tokens, "heads": heads, "head_dim": head_dim,
            "rotated": rotated, "dtype": dtype, "train": train}


def listed():
    return [
        # text stream of a double-stream block: the smallest calls, where launches and host time count
        _norm("text_adaln", "adaln", 1, 256, 3072, "bf16", True),
        _heads("text_qkv", "qkv", 1, 256, 24, 128, 0, "bf16", True),
        # block entry on one context-parallel rank, the residual stream continuing past the norm
        _norm("entry_stream", "stream", 1, 29700, 3072, "bf16", True),
        # attention's gated residual update and the MLP's norm, one of eight ranks
        _norm("gated_rank8", "gated", 1, 14850, 3072, "bf16", True),
        # queries and keys of a double-stream block: every image token rotated
        _heads("qkv_rope", "qkv", 1, 29700, 24, 128, 29700, "bf16", True),
        # single-stream block while sampling: image and text tokens together, text left unrotated, half the heads
        # (two tensor-parallel ranks), forward only
        _heads("qkv_rope_infer", "qkv", 1, 7681, 12, 128, 7425, "bf16", False),
        # four samples with a modulation row each
        _norm("batch_adaln", "adaln", 4, 11056, 3072, "bf16", True),
        # a full 129-frame sequence on one GPU: the largest
        _norm("full_adaln", "adaln", 1, 118800, 3072, "bf16", True),
        # RMSNorm over the hidden dimension in 32 bits
        _norm("rms_fp32", "rms", 2, 4096, 3072, "fp32", True),
        # a smaller model: another hidden size in fp16, a batch of short ragged sequences
        _norm("small_model", "adaln", 8, 1025, 1536, "fp16", True),
        # its attention as the plain module calls it: q as the transposed view of the projection, head dimension 64
        _heads("small_head_view", "view", 2, 2050, 16, 64, 0, "bf16", True),
        # a wider model's hidden size
        _norm("wide_rms", "rms", 1, 6001, 5120, "bf16", True),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["adaln", "adaln", "stream", "gated", "rms", "qkv", "qkv", "view"])
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"])
    train = rng.random() < 0.75
    while True:
        if kind in ("qkv", "view"):
            batch, tokens, heads = rng.choice([1, 1, 2, 4]), _log_int(rng, 64, 60000), rng.choice([6, 8, 12, 16, 24])
            head_dim = 128 if rng.random() < 0.6 else rng.choice([64, 80, 96])
            rotated = 0
            if kind == "qkv" and head_dim == 128 and rng.random() < 0.6:
                rotated = tokens if rng.random() < 0.5 or tokens <= 300 else tokens - rng.randint(1, 256)
            case = {"kind": kind, "batch": batch, "tokens": tokens, "heads": heads, "head_dim": head_dim,
                    "rotated": rotated, "dtype": dtype, "train": train}
        else:
            batch, tokens = rng.choice([1, 1, 2, 3, 4, 8]), _log_int(rng, 64, 118800)
            hidden = 3072 if rng.random() < 0.5 else rng.choice([1024, 1152, 1536, 2048, 2560, 4096])
            if dtype != "fp32" and hidden == 4096 and rng.random() < 0.5:
                hidden = 5120
            case = {"kind": kind, "batch": batch, "tokens": tokens, "hidden": hidden, "dtype": dtype, "train": train}
        if work(case)["bytes"] <= _LARGEST:
            return case


def work(case):
    """Bytes and operations one pass cannot do without: every operand of the forward call and of the backward
    call read once, every result written once.  Row statistics and workspaces are not counted."""
    e, train = _ELEM[case["dtype"]], case["train"]
    kind = case["kind"]
    rows = case["batch"] * case["tokens"]
    if kind in ("qkv", "view"):
        n = rows * case["heads"] * case["head_dim"]
        if kind == "view":  # x, out; dout, x, dx
            return {"bytes": n * e * (5 if train else 2), "flops": n * (12 if train else 4)}
        # forward: q, k in and out (v is a view); backward: three gradients and q, k in, three slices out
        tables = 2 * case["rotated"] * case["head_dim"] * 4
        rot = 12 if case["rotated"] else 0
        return {"bytes": n * e * (12 if train else 4) + tables * (2 if train else 1),
                "flops": 2 * n * ((12 if train else 4) + rot)}
    n = rows * case["hidden"]
    params = case["batch"] * case["hidden"] * e
    if kind == "rms":
        return {"bytes": n * e * (5 if train else 2) + case["hidden"] * e * (3 if train else 1), "flops": n * (12 if train else 4)}
    if kind == "adaln":
        return {"bytes": n * e * (5 if train else 2) + params * (5 if train else 2), "flops": n * (20 if train else 8)}
    if kind == "stream":
        return {"bytes": n * e * (6 if train else 2) + params * (5 if train else 2), "flops": n * (21 if train else 8)}
    return {"bytes": n * e * (10 if train else 4) + params * (8 if train else 3), "flops": n * (27 if train else 10)}


def prepare(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    gen = torch.Generator(device=dev).manual_seed(seed)
    dt = _TYPES[case["dtype"]]
    train = case["train"]

    def rnd(*shape, k=1.0, bias=0.0, dtype=dt):
        t = torch.randn(*shape, device=dev, generator=gen)
        return t.mul_(k).add_(bias).to(dtype)

    def leaf(t):
        return t.requires_grad_(train)

    B, S = case["batch"], case["tokens"]
    state = {"case": case}
    if case["kind"] in ("qkv", "view"):
        H, D = case["heads"], case["head_dim"]
        norms = []
        for _ in range(2 if case["kind"] == "qkv" else 1):
            norm = FL.RMSNorm(D, eps=EPS).to(device=dev, dtype=dt)
            with torch.no_grad():
                norm.weight.copy_(rnd(D, k=0.02, bias=1.0))
            norm.requires_grad_(train)
            norms.append(norm)
        state["norms"] = norms
        state["mixed"] = leaf(rnd(B, S, H, 3 * D))
        state["rotary"] = None
        if case["rotated"]:
            n = case["rotated"]
            angle = torch.outer(torch.arange(n, device=dev, dtype=torch.float32) + float(torch.randint(
                0, 64, (1,), generator=gen, device=dev).item()),
                256.0 ** (-torch.arange(0, D, 2, device=dev, dtype=torch.float32) / D))
            state["rotary"] = tuple(t.repeat_interleave(2, dim=1).contiguous() for t in (angle.cos(), angle.sin()))
        if train:
            state["grads"] = [rnd(B, H, S, D) for _ in range(3 if case["kind"] == "qkv" else 1)]
        return state
    C = case["hidden"]
    state["x"] = leaf(rnd(B, S, C))
    if case["kind"] == "rms":
        norm = FL.RMSNorm(C, eps=EPS).to(device=dev, dtype=dt)
        with torch.no_grad():
            norm.weight.copy_(rnd(C, k=0.02, bias=1.0))
        state["norm"] = norm.requires_grad_(train)
    else:
        state["scale"], state["shift"] = leaf(rnd(B, C, k=0.1)), leaf(rnd(B, C, k=0.1))
    if case["kind"] == "gated":
        state["attn"], state["gate"] = leaf(rnd(B, S, C)), leaf(rnd(B, C, k=0.3))
    if train:
        state["grads"] = [rnd(B, S, C) for _ in range(2 if case["kind"] in ("gated", "stream") else 1)]
    return state


def run(state):
    kind = state["case"]["kind"]
    if kind == "qkv":
        q, k, v = FL.split_qkv_and_norm(state["mixed"], state["norms"][0], state["norms"][1], rotary=state["rotary"])
        outs, leaves = [q, k, v], [state["mixed"], state["norms"][0].weight, state["norms"][1].weight]
    elif kind == "view":
        D = state["case"]["head_dim"]
        query = state["mixed"].detach()[..., :D].transpose(1, 2)
        query.requires_grad_(state["case"]["train"])
        outs, leaves = [state["norms"][0](query)], [query, state["norms"][0].weight]
    elif kind == "rms":
        outs, leaves = [state["norm"](state["x"])], [state["x"], state["norm"].weight]
    elif kind == "adaln":
        leaves = [state["x"], state["scale"], state["shift"]]
        outs = [FL.modulated_layer_norm(*leaves, eps=EPS)]
    elif kind == "stream":
        leaves = [state["x"], state["scale"], state["shift"]]
        outs = list(FL.modulated_layer_norm_keeping_stream(*leaves, eps=EPS))
    else:
        leaves = [state["x"], state["attn"], state["gate"], state["scale"], state["shift"]]
        outs = list(FL.gated_residual_layer_norm(*leaves, eps=EPS))
    if not state["case"]["train"]:
        return outs
    return outs + list(torch.autograd.grad(outs, leaves, state["grads"]))


# About three to four times the distance of the fused path from the same formulas in 64 bits, over the listed and drawn
# kinds at up to 6000 tokens: relative 4.1e-3 / 4.8e-4 / 1.6e-7 and at most 4.2e-2 / 5.4e-3 / 7.3e-7 on one element
# (the gated update's gradient, whose two rounded terms may cancel) in bf16 / fp16 / fp32.  The 32-bit bound leaves
# room for column sums over ten times as many rows in another order.
_BOUNDS = {"bf16": {"rel": 1.2e-2, "max": 0.16}, "fp16": {"rel": 1.8e-3, "max": 0.02}, "fp32": {"rel": 2e-6, "max": 1e-5}}


def tolerance(case):
    return dict(_BOUNDS[case["dtype"]])
