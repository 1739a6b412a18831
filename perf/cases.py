"""What users of this package have it do, as cases that can be timed.

Three programs call the package's public entry points:

* ``bwdbwd``: ``fhog.flash_bwdbwd`` on tensors that a program kept from its forward pass: the call that the package exists for;
* ``hvp``: ``fhog.attention`` differentiated twice by autograd (forward, first backward with ``create_graph=True``, and the
  double-backward): a Hessian-vector product, the core of every step with a penalty on gradients;
* ``step``: ``fhog.attention`` differentiated once: the plain training step of the same model.
"""
import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path.cwd() / "flash-hob_amd"))
import fhog  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _case(program, dtype, B, H, n_q, n_k, d, mask="none", window=0, grad_std=0.1, k_row_scale=False, schedule=""):
    """``mask``: none | causal (n_q == n_k) | bottom_right; ``window``: keys a query sees at most, 0 = all; ``schedule``: as the
    entry points take it, "" = their default."""
    return dict(program=program, dtype=dtype, B=B, H=H, n_q=n_q, n_k=n_k, d=d, mask=mask, window=window, grad_std=grad_std,
                k_row_scale=k_row_scale, schedule=schedule)


def listed():
    return [
        # the smallest use in earnest, a fp32 parity problem of two heads: latency and launches are all it is
        dict(_case("bwdbwd", "fp32", 1, 2, 256, 256, 64, grad_std=1.0), name="fp32_2x256_d64"),
        # a gradient penalty on a short sequence: three entry points of a few launches each behind autograd
        dict(_case("hvp", "bf16", 1, 2, 256, 256, 128, "causal"), name="hvp_bf16_2x256_d128"),
        # one head of the sweep over lengths: too few tiles to fill the chip without splitting the other side
        dict(_case("bwdbwd", "fp16", 1, 1, 8192, 8192, 64), name="fp16_1x8192_d64"),
        # an ordinary encoder layer
        dict(_case("bwdbwd", "bf16", 4, 16, 2048, 2048, 64), name="bf16_64x2048_d64"),
        # an ordinary decoder layer, the shape the package's throughput is quoted on
        dict(_case("bwdbwd", "bf16", 2, 16, 4096, 4096, 128, "causal"), name="bf16_causal_32x4096_d128"),
        # long context, the largest call
        dict(_case("bwdbwd", "bf16", 1, 32, 16384, 16384, 128, "causal"), name="bf16_causal_32x16384_d128"),
        # cross-attention of unequal lengths, keys of widely different norms
        dict(_case("bwdbwd", "bf16", 8, 8, 1024, 8192, 64, k_row_scale=True), name="bf16_cross_64x1024x8192_d64"),
        # ragged lengths under a sliding window: queries that continue a longer context
        dict(_case("bwdbwd", "bf16", 2, 8, 1000, 3001, 128, "bottom_right", 700), name="bf16_window_16x1000x3001_d128"),
        # a training step without second derivatives at the decoder layer's shape
        dict(_case("step", "bf16", 2, 16, 4096, 4096, 128, "causal"), name="step_bf16_32x4096_d128"),
        # second derivatives in single precision at an ordinary size
        dict(_case("hvp", "fp32", 2, 16, 2048, 2048, 128, "causal"), name="hvp_fp32_32x2048_d128"),
        # a gradient penalty under the schedule with the fewest products, odd length
        dict(_case("hvp", "fp16", 4, 12, 1537, 1537, 64, "causal", schedule="three_sweep"), name="hvp_fp16_48x1537_d64"),
        # the small head dim: narrow heads of a small model
        dict(_case("hvp", "bf16", 8, 8, 1024, 1024, 32, "causal"), name="hvp_bf16_64x1024_d32"),
    ]


def _log_between(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    """One more case of the listed ones' ranges: every program, type, head dim and mask; lengths 64 to 16384, odd ones among them;
    1 to 128 heads; at most a fifth of the largest listed case's products (a fortieth of them in single precision or at head dim
    32, which run at a lower rate)."""
    program = rng.choice(["bwdbwd", "bwdbwd", "hvp", "step"])
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"])
    d = rng.choice([64, 128, 64, 128, 32])
    mask = rng.choice(["none", "causal", "causal", "bottom_right"])
    n_q = _log_between(rng, 64, 16384)
    if rng.random() < 0.5:
        n_q = max(64, n_q // 64 * 64)
    n_k = n_q
    if mask == "bottom_right":
        n_k = min(16384, n_q + _log_between(rng, 1, 8192))
    elif mask == "none" and rng.random() < 0.5:
        n_k = _log_between(rng, 64, 16384)
    window = _log_between(rng, 32, max(33, n_k)) if mask != "none" and rng.random() < 0.3 else 0
    slow = dtype == "fp32" or d == 32
    most = 12 * 2 * 128 * 32 * 16384 * 16384 / 2 / (40 if slow else 5)
    per_head = 24 * d * _pairs(n_q, n_k, mask, window)
    heads = max(1, min(128, int(most / per_head)))
    H = rng.choice([1, 2, 8, 12, 16])
    heads = _log_between(rng, 1, heads)
    H = min(H, heads)
    schedule = rng.choice(["", "", "", "fused_stats", "three_sweep"]) if program != "step" else ""
    return _case(program, dtype, max(1, heads // H), H, n_q, n_k, d, mask, window, grad_std=1.0 if dtype == "fp32" else 0.1,
                 schedule=schedule)


def prepare(case, seed):
    dtype, dev = DTYPES[case["dtype"]], torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(int(seed))
    q_shape = (case["B"], case["H"], case["n_q"], case["d"])
    k_shape = (case["B"], case["H"], case["n_k"], case["d"])

    def normal(shape, std=1.0):
        return (torch.randn(shape, generator=g, device=dev) * std).to(dtype)

    std = case["grad_std"]
    q, k, v = normal(q_shape), normal(k_shape), normal(k_shape)
    do, ddq, ddk, ddv = normal(q_shape, std), normal(q_shape, std), normal(k_shape, std), normal(k_shape, std)
    if case["k_row_scale"]:
        k = (k.float() * (torch.rand(k_shape[:3] + (1,), generator=g, device=dev) * 1.5 + 0.5)).to(dtype)
    state = dict(program=case["program"], scale=case["d"] ** -0.5, causal={"none": False, "causal": True}.get(case["mask"], case["mask"]),
                 window=case["window"] or None, schedule=case["schedule"] or None)
    if case["program"] == "bwdbwd":
        o, lse = fhog.attention_forward(q, k, v, state["scale"], state["causal"], window=state["window"])
        state["tensors"] = (q, k, v, o, do, ddq, ddk, ddv, lse)
    else:
        leaves = (q, k, v, do) if case["program"] == "hvp" else (q, k, v)
        for t in leaves:
            t.requires_grad_(True)
        state.update(leaves=(q, k, v), do=do, directions=(ddq, ddk, ddv))
    return state


def run(state):
    if state["program"] == "bwdbwd":
        return fhog.flash_bwdbwd(*state["tensors"], state["scale"], causal=state["causal"], window=state["window"], schedule=state["schedule"])
    q, k, v = state["leaves"]
    out = fhog.attention(q, k, v, state["causal"], state["window"], state["schedule"])
    if state["program"] == "step":
        return (out, *torch.autograd.grad(out, (q, k, v), state["do"]))
    first = torch.autograd.grad(out, (q, k, v), state["do"], create_graph=True)
    second = torch.autograd.grad(first, (q, k, v, state["do"]), state["directions"])
    return (out, *first, *second)


def _pairs(n_q, n_k, mask, window):
    """(query, key) pairs of one head that the mask leaves visible."""
    if mask == "none":
        return n_q * n_k
    shift = n_k - n_q if mask == "bottom_right" else 0
    return sum(min(i + shift + 1, window or n_k) for i in range(n_q))


def work(case):
    """The materialised formula's contractions (2 forward, 5 in the first backward, 12 in the double-backward) over the visible
    pairs, and every tensor once."""
    heads, d, program = case["B"] * case["H"], case["d"], case["program"]
    pairs = heads * _pairs(case["n_q"], case["n_k"], case["mask"], case["window"])
    products = {"bwdbwd": 12, "hvp": 2 + 5 + 12, "step": 2 + 5}[program]
    q_side, k_side = {"bwdbwd": (4 + 2, 4 + 2),      # Q O dO ddQ dQ2 ddO | K V ddK ddV dK2 dV2
                      "hvp": (3 + 4, 4 + 4),         # Q dO ddQ, O dQ dQ2 ddO | K V ddK ddV, dK dV dK2 dV2
                      "step": (2 + 2, 2 + 2)}[program]
    es = DTYPES[case["dtype"]].itemsize
    nbytes = heads * d * es * (q_side * case["n_q"] + k_side * case["n_k"])
    if program == "bwdbwd":
        nbytes += heads * case["n_q"] * 4            # the log-sum-exp
    return {"bytes": nbytes, "flops": 2 * d * pairs * products}


def tolerance(case):
    """About four times the largest error against the same sums in double precision, over all outputs and the shapes above up to
    8192 x 8192 (relative error, largest single one): bf16 2.6e-3 and 5.8e-2, fp16 6.4e-4 and 8e-3, fp32 1.5e-6 and 1.9e-5. The
    largest single errors sit in the first rows of a causal mask."""
    return {"bf16": {"rel": 1e-2, "max": 0.25}, "fp16": {"rel": 2.5e-3, "max": 4e-2}, "fp32": {"rel": 6e-6, "max": 1e-4}}[case["dtype"]]
