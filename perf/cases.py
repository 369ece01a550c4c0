"""The work whose speed counts: one causal linear-attention operator, seen from its public entry
points.

Five ways in: the autograd function ``causal_dot_product`` (training step, or forward alone), its
stateful form ``causal_dot_product_with_state`` (a piece of a prompt; one step of decoding), the
module ``CausalLinearAttention`` (eval and training) and the encoder built around it.  Sizes are
those of ``bench.py``'s workloads and of the tests, plus generic ones between them.

Every case is a dict of plain values: ``kind`` (which way in), ``N`` sequences, ``H`` heads, ``L``
positions, ``E`` and ``M`` widths of a query and of a value row, ``dtype`` of the rows.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.abspath("fast-transformers_amd"))

from fast_transformers_amd.attention import CausalLinearAttention, build_causal_linear_encoder  # noqa: E402
from fast_transformers_amd.causal_product import causal_dot_product, causal_dot_product_with_state  # noqa: E402
from fast_transformers_amd.masking import LengthMask, TriangularCausalMask  # noqa: E402

_DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16}


def _case(kind, N, H, L, E, M, dtype="fp32", **more):
    return dict(kind=kind, N=N, H=H, L=L, E=E, M=M, dtype=dtype, **more)


def listed():
    return [
        # one token for each of 32 sequences being generated: launches and latency only
        dict(_case("decode", 32, 8, 1, 64, 64), name="decode_step"),
        # the smallest forward that the benchmark knows: a few short sequences in inference
        dict(_case("forward", 2, 4, 512, 64, 64), name="forward_small"),
        # the next 2048 tokens of four half-precision prompts, state handed in and out
        dict(_case("prefill", 4, 16, 2048, 64, 64, "bf16"), name="prefill_bf16"),
        # the operator's training step at its quick-start size (the headline)
        dict(_case("train", 10, 8, 1000, 64, 64), name="train_quickstart"),
        # the same step with half-precision rows
        dict(_case("train", 10, 8, 1000, 64, 64, "bf16"), name="train_bf16"),
        # odd widths, a length that divides nothing, chains that fill the GPU unevenly
        dict(_case("train", 9, 11, 1531, 25, 33), name="train_odd_widths"),
        # wide heads, full batch
        dict(_case("train", 8, 16, 4096, 128, 128), name="train_wide"),
        # one very long sequence (the carried state over 65536 positions)
        dict(_case("train", 1, 16, 65536, 64, 64), name="train_long"),
        # half-precision rows, narrow keys, wide values: the most memory traffic
        dict(_case("train", 4, 32, 16384, 32, 128, "bf16"), name="train_bf16_wide_values"),
        # the attention module in inference over a padded batch
        dict(_case("attention", 10, 8, 1000, 64, 64, ragged=True), name="attention_eval_ragged"),
        # the attention module's training step at the encoder's size
        dict(_case("attention_train", 10, 8, 4096, 64, 64, ragged=False), name="attention_train"),
        # the eight-layer encoder's forward: the operator as part of a model
        dict(_case("encoder", 10, 8, 4096, 64, 64, layers=8, feed_forward=1024), name="encoder_eval"),
    ]


def _spread(rng, low, high):
    """A whole number between low and high, even over its logarithm."""
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _widths(rng):
    """(E, M): mostly the usual head sizes, sometimes unusual or odd ones."""
    r = rng.random()
    if r < 0.55:
        w = rng.choice([32, 64, 64, 128])
        return w, w
    if r < 0.7:
        return rng.choice([32, 64, 128]), rng.choice([32, 64, 128])
    if r < 0.85:
        return 4 * rng.randint(4, 32), 4 * rng.randint(4, 32)
    return rng.randint(10, 128), rng.randint(10, 128)


# no drawn operator call moves more bytes than the long training step, and none multiplies more
# than the wide one
_MOST_BYTES = 3.0e9
_MOST_FLOPS = 1.25e11


def draw(rng):
    kind = rng.choice(["train", "train", "train", "train", "forward", "prefill", "decode",
                       "attention", "attention_train", "encoder"])
    while True:
        dtype = "bf16" if rng.random() < 0.3 else "fp32"
        H = rng.choice([1, 4, 8, 8, 12, 16, 32])
        if kind in ("train", "forward"):
            E, M = _widths(rng)
            case = _case(kind, _spread(rng, 1, 64), H, _spread(rng, 64, 65536), E, M, dtype)
        elif kind == "prefill":
            w = rng.choice([32, 64, 64, 128])
            case = _case(kind, _spread(rng, 1, 16), H, _spread(rng, 16, 8192), w, w, dtype)
        elif kind == "decode":
            w = rng.choice([32, 64, 64, 128])
            case = _case(kind, _spread(rng, 1, 256), H, 1, w, w, dtype)
        elif kind in ("attention", "attention_train"):
            w = rng.choice([32, 64, 64, 64, 128])
            case = _case(kind, _spread(rng, 1, 32), H, _spread(rng, 64, 8192), w, w,
                         ragged=rng.random() < 0.5)
        else:
            w = rng.choice([32, 64, 64])
            case = _case(kind, _spread(rng, 1, 10), rng.choice([4, 8, 8]), _spread(rng, 64, 4096), w, w,
                         layers=rng.randint(2, 8), feed_forward=rng.choice([512, 1024, 1024]))
        w = work(case)
        if kind == "encoder" or (w["bytes"] <= _MOST_BYTES and w["flops"] <= _MOST_FLOPS):
            return case


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    N, H, L, E, M = (case[k] for k in "NHLEM")
    dtype = _DTYPES[case["dtype"]]

    def normal(*shape):
        return torch.randn(*shape, device="cuda", generator=gen)

    kind = case["kind"]
    if kind == "encoder":
        # random weights of the architecture, uniform inputs, as the encoder's workload has them
        torch.manual_seed(seed)
        with torch.device("cuda"):
            model = build_causal_linear_encoder(
                n_layers=case["layers"], n_heads=H, query_dimensions=E, value_dimensions=M,
                feed_forward_dimensions=case["feed_forward"]).eval()
        x = torch.rand(N, L, H * M, device="cuda", generator=gen)
        return {"kind": kind, "model": model, "x": x, "mask": TriangularCausalMask(L, device="cuda")}
    if kind in ("attention", "attention_train"):
        # raw projections, both signs, in the module's (N, L, H, X) layout
        q, k, v, g = (normal(N, L, H, w) for w in (E, E, M, M))
        lengths = torch.full((N,), L, dtype=torch.int64, device="cuda")
        if case["ragged"]:
            lengths = torch.randint((L + 1) // 2, L + 1, (N,), device="cuda", generator=gen)
        lengths = LengthMask(lengths, max_len=L)
        if kind == "attention_train":
            q, k, v = (t.requires_grad_(True) for t in (q, k, v))
        return {"kind": kind, "attention": CausalLinearAttention(E), "q": q, "k": k, "v": v, "g": g,
                "mask": TriangularCausalMask(L, device="cuda"), "lengths": lengths}
    # the operator sees mapped queries and keys: elu(x) + 1, positive
    q, k = ((torch.nn.functional.elu(normal(N, H, L, E)) + 1).to(dtype) for _ in range(2))
    v = normal(N, H, L, M).to(dtype)
    state = {"kind": kind, "q": q, "k": k, "v": v}
    if kind == "train":
        for t in (q, k, v):
            t.requires_grad_(True)
        state["g"] = normal(N, H, L, M)
    if kind in ("prefill", "decode"):
        # what a few hundred earlier positions leave behind
        state["s"] = 20 * normal(N, H, E, M)
    return state


def run(state):
    kind = state["kind"]
    if kind == "train":
        inputs = (state["q"], state["k"], state["v"])
        out = causal_dot_product(*inputs)
        return (out.detach(),) + torch.autograd.grad(out, inputs, state["g"])
    if kind == "attention_train":
        inputs = (state["q"], state["k"], state["v"])
        out = state["attention"](*inputs, state["mask"], state["lengths"], state["lengths"])
        return (out.detach(),) + torch.autograd.grad(out, inputs, state["g"])
    with torch.no_grad():
        if kind == "forward":
            return causal_dot_product(state["q"], state["k"], state["v"])
        if kind in ("prefill", "decode"):
            return causal_dot_product_with_state(state["q"], state["k"], state["v"], state["s"])
        if kind == "attention":
            return state["attention"](state["q"], state["k"], state["v"], state["mask"],
                                      state["lengths"], state["lengths"])
        return state["model"](state["x"], attn_mask=state["mask"])


def work(case):
    """Forward: Q, K, V read and the product written, 4 E M operations per position.  Backward:
    those and the gradient read (the product's consumer has run in between), three gradients
    written, 10 E M operations."""
    N, H, L, E, M = (case[k] for k in "NHLEM")
    rows = N * H * L
    size = 2 if case["dtype"] == "bf16" else 4
    inputs, result = (2 * E + M) * size, 4 * M
    kind = case["kind"]
    if kind == "encoder":
        d, f = H * M, case["feed_forward"]
        weights = case["layers"] * (2 * d * H * E + 2 * d * d + 2 * d * f)
        per_token = case["layers"] * H * 4 * E * M + 2 * weights
        return {"bytes": 4 * (2 * N * L * d + weights), "flops": N * L * per_token}
    if kind in ("train", "attention_train"):
        # the module's backward also needs the forward's result and its denominators (one a row)
        more = (4 * M + 8) if kind == "attention_train" else 0
        return {"bytes": rows * (3 * inputs + 2 * result + more), "flops": rows * 14 * E * M}
    states = 2 * 4 * N * H * E * M if kind in ("prefill", "decode") else 0
    return {"bytes": rows * (inputs + result) + states, "flops": rows * 4 * E * M}


def tolerance(case):
    # Four times the distance from an evaluation of the same path in float64: at most 1.3e-6
    # (2-norm) and 5.6e-5 (largest) for float32 results over all the kinds, 1.7e-3 and 3.9e-3
    # (half a unit in the last place) for gradients of bf16 rows.
    if case["dtype"] == "bf16" and case["kind"] == "train":
        return {"rel": 7e-3, "max": 1.6e-2}
    return {"rel": 5e-6, "max": 2.5e-4}
