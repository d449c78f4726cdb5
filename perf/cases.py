"""Workloads of the MoE layer whose speed is watched.

A case is one thing that a sampler of a DiT-MoE model does with a layer of this
package: a call of a block (plain, fused with the norm / modulation / residual
around it), a pair of steps with the skip cache, a few step-lagged steps, or the
routed experts on a caller's own routing.  ``listed()`` are fixed ones, ``draw``
makes more of the same ranges, ``prepare`` builds a block and its inputs on the
GPU, ``run`` is one pass through the public entry points.
"""
import math

import torch

from dice_amd import ParaMode, SparseMoeBlock, diep
from dice_amd.ep_fwd import moe_infer_ep

DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}

# Fields of a case:
#   width, experts            the block's hidden size and routed experts (top-2, expert width 4 x hidden)
#   variant                   swiglu (shared expert of width 2 x hidden) or gelu_tanh (two shared experts of the routed shape)
#   dtype                     of activations and weights
#   fp8                       none, weights (e4m3 experts, 16-bit activations), rows (activations too, one scale per row),
#                             blocks (h quantised in blocks of 32 columns)
#   samples, tokens           the batch [samples, tokens, width]
#   call                      forward, modulated (x + gate * moe(modulate(norm(x)))), skip (a full step that fills the skip
#                             cache, then a step that reads it), lagged (a synchronous step, then three displaced ones),
#                             routed (moe_infer_ep on given routing)
#   skip_mode                 which routed slot a skip step leaves out
#   zipf                      exponent of the expert load set through the router bias, 0 for an even load
#   renorm                    routing weights renormalised over the top 2


def _case(width, experts, variant, dtype, samples, tokens, call="forward", fp8="none", zipf=0.0, renorm=False,
          skip_mode="high"):
    return dict(width=width, experts=experts, variant=variant, dtype=dtype, fp8=fp8, samples=samples, tokens=tokens,
                call=call, skip_mode=skip_mode, zipf=zipf, renorm=renorm)


def listed():
    return [
        # One 256-pixel image through DiT-S, which is served in fp32: the smallest call, all latency.
        dict(_case(384, 8, "swiglu", "f32", 1, 256), name="s_f32_one_image"),
        # The DiT-S benchmark block: four images, GELU experts, weights renormalised over the top 2.
        dict(_case(384, 8, "gelu_tanh", "f32", 4, 256, renorm=True), name="s_f32_four_images"),
        # A sampling batch of 16 images with guidance (twice the rows) through DiT-B in fp32.
        dict(_case(768, 8, "swiglu", "f32", 32, 256, "modulated"), name="b_f32_batch"),
        # One image with guidance through DiT-XL in half precision: interactive sampling, as a DiT block calls the layer.
        dict(_case(1152, 8, "swiglu", "f16", 2, 256, "modulated"), name="xl_f16_one_image"),
        # The headline DiT-XL block: 16 images with guidance.
        dict(_case(1152, 8, "swiglu", "bf16", 32, 256), name="xl_bf16_batch"),
        # The same batch with two-matrix GELU experts and two shared experts of the routed shape, fused into its caller.
        dict(_case(1152, 8, "gelu_tanh", "bf16", 32, 256, "modulated"), name="xl_bf16_gelu_batch"),
        # 512-pixel images and a skewed expert load.
        dict(_case(1152, 8, "swiglu", "bf16", 16, 1024, zipf=1.2), name="xl_bf16_512px_zipf"),
        # Conditional communication: a full step and a skip step of the staleness schedule.
        dict(_case(1152, 8, "swiglu", "bf16", 32, 256, "skip"), name="xl_bf16_skip_pair"),
        # Displaced steps of a small batch with an odd number of tokens per sample.
        dict(_case(1152, 8, "swiglu", "f16", 6, 333, "lagged"), name="xl_f16_lagged_odd"),
        # Routed experts on a caller's own routing, DiT-G as it is served (width 1408, fp16), a ragged batch.
        dict(_case(1408, 16, "swiglu", "f16", 7, 301, "routed"), name="g_f16_routed_odd"),
        # The DiT-G benchmark block: fp8 experts and activations on the fp8 matrix pipe.
        dict(_case(2048, 16, "swiglu", "bf16", 32, 256, fp8="rows"), name="g_fp8_batch"),
        # One image with guidance through the same block with fp8 weights only: weight streaming.
        dict(_case(2048, 16, "swiglu", "bf16", 2, 256, fp8="weights"), name="g_w8_one_image"),
    ]


# The blocks that draw() picks from: width, experts, types, fp8 forms, most tokens of a call.
_BLOCKS = [
    (384, 8, ("f32",), ("none",), 8192),
    (768, 8, ("f32",), ("none",), 8192),
    (1152, 8, ("bf16", "f16"), ("none",), 16384),
    (1152, 8, ("bf16", "f16"), ("none",), 8192),
    (1408, 16, ("f16",), ("none",), 4096),
    (2048, 16, ("bf16",), ("weights", "rows", "blocks"), 8192),
]


def draw(rng):
    width, experts, dtypes, fp8s, most = rng.choice(_BLOCKS)
    variant = rng.choice(("swiglu", "swiglu", "gelu_tanh"))
    call = rng.choice(("forward", "forward", "modulated", "modulated", "skip", "lagged", "routed"))
    total = int(round(math.exp(rng.uniform(math.log(256), math.log(most)))))
    tokens = rng.choice((256, 256, 1024, rng.randint(65, 513)))
    tokens = min(tokens, total)
    samples = max(1, total // tokens)
    case = _case(width, experts, variant, rng.choice(dtypes), samples, tokens, call, rng.choice(fp8s),
                 rng.choice((0.0, 0.0, 1.2)), rng.choice((False, False, True)), rng.choice(("high", "low")))
    time, flops = max(_cost(c) for c in listed()), max(work(c)["flops"] for c in listed())
    while case["samples"] > 1 and (_cost(case) > time or work(case)["flops"] > flops):
        case["samples"] //= 2
    return case


# --------------------------------------------------------------------------- #


class State:
    """What a user's program keeps between calls: the block and this step's inputs."""

    def __init__(self, case, block, **inputs):
        self.call, self.block = case["call"], block
        self.__dict__.update(inputs)


def prepare(case, seed):
    dev = torch.device("cuda")
    dtype = DTYPES[case["dtype"]]
    width, experts, call = case["width"], case["experts"], case["call"]
    gen = torch.Generator(dev).manual_seed(seed)

    def normal(*shape, std=1.0):
        return torch.randn(*shape, generator=gen, device=dev).mul_(std).to(dtype)

    mode = ParaMode(ep=call in ("skip", "lagged"), ep_async=call == "lagged", ep_async_mode="all")
    with torch.device(dev):
        block = SparseMoeBlock(width, 4, experts, 2, pretraining_tp=1, layer_idx=0, total_layers=1, para_mode=mode,
                               variant=case["variant"], n_shared_experts=2 if case["variant"] == "swiglu" else 8)
    block = block.to(dtype=dtype).eval()
    with torch.no_grad():
        for name, p in block.named_parameters():
            if name == "gate.weight":          # router N(0, 0.02)
                p.copy_(normal(*p.shape, std=0.02))
            elif p.dim() == 2:                 # experts Xavier-uniform
                bound = math.sqrt(6.0 / (p.shape[0] + p.shape[1]))
                p.copy_(torch.rand(p.shape, generator=gen, device=dev).mul_(2 * bound).sub_(bound))
            else:                              # biases of the GELU experts
                p.copy_(normal(*p.shape, std=0.02))
    block.gate.norm_topk_prob = case["renorm"]
    if case["zipf"]:
        load = torch.tensor([(e + 1.0) ** -case["zipf"] for e in range(experts)], device=dev)
        block.gate.bias = (load / load.sum()).log().float()
    if case["fp8"] == "none":
        block.pack_weights()
    else:
        block.quantize_fp8(activations=case["fp8"] != "weights", h_blocks=case["fp8"] == "blocks")

    shape = (case["samples"], case["tokens"], width)
    n = shape[0] * shape[1]
    if call == "modulated":
        return State(case, block, x=normal(*shape), shift=normal(shape[0], width, std=0.2),
                     scale=normal(shape[0], width, std=0.2), gate=normal(shape[0], width, std=0.5))
    if call == "routed":
        logits = torch.randn(n, experts, generator=gen, device=dev)
        if case["zipf"]:
            logits += block.gate.bias
        weight, index = logits.softmax(-1).topk(2, dim=-1, sorted=False)
        return State(case, block, x=normal(n, width), index=index.reshape(-1).contiguous(),
                     weight=weight.reshape(-1, 1).to(dtype).contiguous())
    if call in ("skip", "lagged"):
        # Consecutive steps of a sampler: the input drifts a little from one to the next.
        xs = [normal(*shape)]
        for _ in range(1 if call == "skip" else 3):
            xs.append((xs[-1].float() + 0.05 * normal(*shape).float()).to(dtype))
        if call == "skip":
            diep.ep_cache_init(1, noskip_step=2, skip_mode=case["skip_mode"])
        else:
            diep.ep_cache_init(1)
            diep.use_latest_expert_weights(False)
        return State(case, block, xs=xs)
    return State(case, block, x=normal(*shape))


def run(state):
    block = state.block
    if state.call == "forward":
        return block(state.x)
    if state.call == "modulated":
        return block.forward_modulated(state.x, state.shift, state.scale, state.gate)
    if state.call == "routed":
        return moe_infer_ep(state.x, block.experts, state.index, state.weight, 2, False)
    diep.ep_cache_clear()
    if state.call == "skip":
        diep.ep_set_step(2)
        full = block(state.xs[0])
        diep.ep_set_step(1)
        return full, block(state.xs[1])
    diep.diep_force_sync()
    out = [block(state.xs[0])]
    diep.diep_cancel_sync()
    return out + [block(x) for x in state.xs[1:]]


# --------------------------------------------------------------------------- #


def _calls(case):
    """(calls of a pass, routed slots of all of them per token)."""
    return {"skip": (2, 3), "lagged": (4, 8)}.get(case["call"], (1, 2))


def _matrices(case):
    """(elements of one routed expert, elements of the shared expert)."""
    d, up = case["width"], 2 if case["variant"] == "swiglu" else 1
    shared = 2 * d if case["variant"] == "swiglu" else 8 * d
    return (up + 1) * d * 4 * d, 0 if case["call"] == "routed" else (up + 1) * d * shared


def _flops(case):
    """Multiply-adds x 2 of (routed experts, everything else)."""
    n, (calls, slots), (routed, shared) = case["samples"] * case["tokens"], _calls(case), _matrices(case)
    router = 0 if case["call"] == "routed" else case["width"] * case["experts"]
    return 2.0 * n * slots * routed, 2.0 * n * calls * (shared + router)


def work(case):
    n, d = case["samples"] * case["tokens"], case["width"]
    es = DTYPES[case["dtype"]].itemsize
    routed, shared = _matrices(case)
    weights = case["experts"] * routed * (es if case["fp8"] == "none" else 1) + shared * es + case["experts"] * d * es
    rows = 2 * _calls(case)[0] * n * d * es          # each call's input and output
    if case["call"] == "skip":
        rows += 2 * n * d * es                       # the cache is written and read
    if case["call"] == "modulated":
        rows += 3 * case["samples"] * d * es
    if case["call"] == "routed":
        rows += 2 * n * (8 + es)
    return {"bytes": weights + rows, "flops": sum(_flops(case))}


def _cost(case):
    """Time of the operations at nominal rates: what draw() bounds."""
    routed, rest = _flops(case)
    rate = {"f32": 157e12, "f16": 2500e12, "bf16": 2500e12}[case["dtype"]]
    return routed / (5000e12 if case["fp8"] in ("rows", "blocks") else rate) + rest / rate


def tolerance(case):
    if case["fp8"] in ("rows", "blocks"):
        return {"rel": 2e-2}   # an e4m3 code that rounds the other way moves its product by up to 1/16
    # fp32 sums of up to 3072 products; h and y rounded to 11 or 8 bits
    return {"rel": {"f32": 1e-5, "f16": 2e-3, "bf16": 1e-2}[case["dtype"]]}
