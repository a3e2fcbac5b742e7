"""The work a user of chill_attention has it do, as cases that can be timed and compared.

A case names a mask, the shape of one attention layer and the pass a program takes through it: "training" is
the forward and the three gradients, "forward" the output alone (inference), "forward_lse" the output and LSE2 (what a
caller needs who merges several partial attentions).  `listed` holds twelve fixed cases, `draw` gives others of the same
ranges: every mask of the package, head dims 64 to 256, the three element types, sequences of 128 to 16384 rows, most of
them not a multiple of any tile, one to 32 heads with and without shared key / value heads, padded batches, and both
storage orders of the heads.
"""

import math
import os
import sys

import torch

# the package lies one folder below the repository's root, which is the working folder
sys.path.insert(0, os.path.abspath("chill-attention_amd"))

import chill_attention as ca  # noqa: E402

DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


def case(name, mask, args, dtype, B, H, H_kv, T, D, work="training", sigma=1.0, padded=False, layout="bhtd"):
    a0, a1 = (tuple(args) + (0, 0))[:2]
    return {"name": name, "mask": mask, "a0": a0, "a1": a1, "dtype": dtype, "B": B, "H": H, "H_kv": H_kv, "T": T, "D": D,
            "work": work, "sigma": sigma, "padded": padded, "layout": layout}


def listed():
    return [
        # the smallest call: a short prompt through a small fp32 model, where the launch and the host decide
        case("causal_f32_small_forward", "Causal", (), "f32", 1, 2, 2, 256, 64, work="forward"),
        # a training step of a small model on one short sequence: host work, autograd and three launches
        case("causal_short_training", "Causal", (), "bf16", 1, 8, 8, 512, 64),
        # local attention of a long-document encoder
        case("sliding_window_training", "SlidingWindow", (128, 128), "bf16", 4, 16, 16, 4096, 64),
        # the headline: a decoder layer of a large language model in training
        case("causal_training", "Causal", (), "bf16", 8, 16, 16, 8192, 128),
        # block-wise streaming attention (speech) over a long recording
        case("chunkwise_training", "Chunkwise", (128, 2), "f16", 2, 32, 32, 16384, 128, sigma=0.5),
        # a prefix language model: bidirectional prompt, causal continuation
        case("prefix_lm_training", "PrefixLM", (1024,), "bf16", 4, 32, 32, 8192, 64),
        # the same mask at full fp32 precision
        case("prefix_lm_f32_training", "PrefixLM", (1024,), "f32", 1, 8, 8, 2048, 64),
        # prefill of one long prompt: one GPU's share of the heads, a shared key / value head, heads interleaved in
        # storage as a fused projection leaves them
        case("causal_prefill_few_heads", "Causal", (), "bf16", 1, 8, 1, 8192, 128, work="forward", layout="bthd"),
        # fine-tuning on a padded batch of sentences of different lengths, grouped key / value heads
        case("causal_padded_gqa_training", "Causal", (), "bf16", 4, 32, 8, 2085, 128, padded=True, layout="bthd"),
        # a bidirectional encoder on sequences of no round length
        case("full_ragged_training", "Full", (), "f16", 8, 12, 12, 4042, 64),
        # a narrow window (benchmark/benchmark.py's): a few keys per row, nearly all traffic
        case("narrow_window_training", "SlidingWindow", (16, 16), "f16", 8, 4, 4, 6000, 128),
        # the widest heads
        case("causal_wide_heads_training", "Causal", (), "bf16", 4, 8, 8, 8192, 256),
    ]


def _size(rng, lo, hi):
    """A length between lo and hi, spread over its logarithm; one in three is a multiple of 128."""
    n = round(math.exp(rng.uniform(math.log(lo), math.log(hi))))
    return max(lo, n // 128 * 128) if rng.random() < 1 / 3 else n


def _cost(c):
    """Seconds one pass should take, roughly: enough to keep drawn cases below the largest listed one."""
    w = work(c)
    # a row of a narrow band still takes whole tiles of keys
    tiles = 4.0 * c["B"] * c["H"] * c["T"] * 128 * c["D"] * (3.5 if c["work"] == "training" else 1.0)
    rate = 5e13 if c["dtype"] == "f32" else 6e14
    return (w["flops"] + tiles) / rate + w["bytes"] / 2e12


def draw(rng):
    most = _cost(listed()[3])
    while True:
        mask = rng.choice(["Full", "Causal", "Causal", "SlidingWindow", "Chunkwise", "PrefixLM"])
        T = _size(rng, 128, 16384)
        if mask == "SlidingWindow":
            args = (_size(rng, 16, 1024), rng.choice([0, 16, 128, _size(rng, 16, 512)]))
        elif mask == "Chunkwise":
            args = (rng.choice([16, 100, 128, _size(rng, 16, 512)]), rng.choice([0, 1, 2, 4, 8]))
        elif mask == "PrefixLM":
            args = (min(T, _size(rng, 128, 2048)),)
        else:
            args = ()
        D = rng.choice([64, 64, 128, 128, 128, 256])
        dtype = rng.choice(["bf16", "bf16", "f16", "f32"]) if D < 256 else rng.choice(["bf16", "f16"])
        H = rng.choice([2, 4, 8, 12, 16, 32])
        H_kv = H // rng.choice([g for g in (1, 1, 2, 4, 8) if H % g == 0])
        B = rng.choice([1, 1, 2, 4, 8])
        c = case("", mask, args, dtype, B, H, H_kv, T, D, work=rng.choice(["training", "training", "forward", "forward_lse"]),
                 sigma=rng.choice([0.5, 1.0, 1.0]), padded=B > 1 and rng.random() < 0.3, layout=rng.choice(["bhtd", "bthd"]))
        del c["name"]
        if _cost(c) <= 0.6 * most:
            return c


def _mask(c):
    name = c["mask"] + "ChillMask"
    count = {"SlidingWindow": 2, "Chunkwise": 2, "PrefixLM": 1}.get(c["mask"], 0)
    return getattr(ca, name)(*(c["a0"], c["a1"])[:count])


def _lengths(c):
    """The valid lengths of a padded batch: spread evenly from a quarter of T to all of it."""
    if not c["padded"]:
        return [c["T"]] * c["B"]
    return [max(1, round(c["T"] * (0.25 + 0.75 * (i + 1) / c["B"]))) for i in range(c["B"])]


def prepare(c, seed):
    g = torch.Generator("cuda").manual_seed(seed)

    def tensor(heads):
        B, T, D = c["B"], c["T"], c["D"]
        shape = (B, heads, T, D) if c["layout"] == "bhtd" else (B, T, heads, D)
        x = (torch.randn(shape, device="cuda", generator=g) * c["sigma"]).to(DTYPES[c["dtype"]])
        return x if c["layout"] == "bhtd" else x.transpose(1, 2)

    training = c["work"] == "training"
    q, k, v = (tensor(h).requires_grad_(training) for h in (c["H"], c["H_kv"], c["H_kv"]))
    lens = None
    if c["padded"]:
        order = torch.randperm(c["B"], device="cuda", generator=g)
        lens = torch.tensor(_lengths(c), dtype=torch.int32, device="cuda")[order]
    d_out = tensor(c["H"]) if training else None
    return {"q": q, "k": k, "v": v, "d_out": d_out, "lens": lens, "mask": _mask(c), "work": c["work"]}


def run(s):
    q, k, v = s["q"], s["k"], s["v"]
    if s["work"] == "training":
        out = ca.chill_attention(q, k, v, mask=s["mask"], lens=s["lens"])
        dq, dk, dv = torch.autograd.grad(out, (q, k, v), s["d_out"])
        return {"out": out.detach(), "dq": dq, "dk": dk, "dv": dv}
    with torch.no_grad():
        if s["work"] == "forward_lse":
            out, lse = ca.chill_attention(q, k, v, mask=s["mask"], lens=s["lens"], return_lse=True)
            return {"out": out, "lse": lse}
        return {"out": ca.chill_attention(q, k, v, mask=s["mask"], lens=s["lens"])}


def work(c):
    """4 * D operations per visible score entry and head forward, 2.5 times that for the gradients; every input
    row within its sequence read once, every output row written once."""
    mask, lengths = _mask(c), _lengths(c)
    entries = sum(mask.nnz(n) for n in lengths)
    training = c["work"] == "training"
    es = 4 if c["dtype"] == "f32" else 2
    rows_read, rows_written = sum(lengths), c["B"] * c["T"]
    read = rows_read * (c["H"] * (2 if training else 1) + 2 * c["H_kv"])
    written = rows_written * (c["H"] * (2 if training else 1) + (2 * c["H_kv"] if training else 0))
    lse = 4 * rows_written * c["H"] if c["work"] == "forward_lse" else 0
    return {"bytes": (read + written) * c["D"] * es + lse, "flops": int(4 * c["H"] * c["D"] * entries * (3.5 if training else 1))}


# Relative errors (2-norm, and the largest difference over the larger of the value and the root mean square) of two
# correct implementations.  This path against attention in 64 bits, the largest seen over masks, head dims, lengths of
# 128 to 3000 rows and both sigmas: f32 2.2e-6 and 3.9e-5, f16 3.6e-4 and 7.2e-3, bf16 2.9e-3 and 9.5e-2; four times that.
TOLERANCE = {
    "f32": {"rel": 9e-6, "max": 1.6e-4},
    "f16": {"rel": 1.5e-3, "max": 3e-2},
    "bf16": {"rel": 1.2e-2, "max": 4e-1},
}


def tolerance(c):
    return TOLERANCE[c["dtype"]]
