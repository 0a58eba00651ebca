"""The work that a user of the MoE layer has it do, as cases that can be timed.

A case is a plain dict:

  task            "infer"     MoE module in eval mode under no_grad: a decode step or a prefill chunk
                  "train"     MoE module, forward and backward of the output and of the load-balancing loss
                  "rounding"  router GEMM, token-rounding router, general-routing entry; forward only or with backward
  backward        whether the pass includes the backward pass
  T H I E K       tokens, hidden size, expert width, experts, experts per token
  dtype act bias  element type, activation, whether the layer has biases
  skew            False: balanced router; True: expert popularity follows Zipf's law
  fp8             block-scaled fp8 operands: in the forward, and with a backward pass in the activation gradients too

Sizes are those of the configurations in bench.py and in the tests; the ragged ones are any multiples of 64.
"""

import math
import os
import sys
from contextlib import ExitStack

import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.abspath("sonic-moe_amd"))  # the repository's root is the working folder

from sonicmoe import MoE, enable_fp8_backward, enable_fp8_forward, moe_general_routing_inputs  # noqa: E402
from sonicmoe.enums import ActivationType, is_glu  # noqa: E402
from sonicmoe.functional.fp8 import cache_quantized_weights  # noqa: E402
from sonicmoe.routing import token_choice_rounding  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}

# (H, I, E, K): layers of the benchmark configurations and of the tests
MODELS = [
    (512, 256, 8, 2),
    (768, 256, 128, 8),
    (1536, 256, 128, 8),
    (1536, 512, 64, 4),
    (1536, 1024, 32, 2),
    (4096, 256, 256, 16),
    (4096, 512, 128, 8),
    (4096, 1024, 64, 4),
    (4096, 1024, 128, 8),
    (4096, 1536, 128, 8),
]
GATED = ["swiglu", "geglu", "reglu"]
UNGATED = ["relu_sq", "relu", "gelu", "silu"]
ROUNDING_TILE = 128
AUX_COEFFICIENT = 0.01  # weight of the load-balancing loss in the training loss


def _case(task, T, model, *, backward=None, dtype="bf16", act="swiglu", bias=False, skew=False, fp8=False, **more):
    H, I, E, K = model
    return dict(more, task=task, backward=task == "train" if backward is None else backward, T=T, H=H, I=I, E=E, K=K,
                dtype=dtype, act=act, bias=bias, skew=skew, fp8=fp8)


def listed():
    return [
        # one sequence being decoded: latency, launches, and the weights of K experts
        _case("infer", 1, (4096, 1024, 128, 8), name="decode_1"),
        # a serving batch in decode: half the experts' weights and more are read for a few rows each
        _case("infer", 64, (4096, 1024, 128, 8), name="decode_64"),
        # a smaller layer's decode batch, odd size, fp16 weights
        _case("infer", 23, (1536, 256, 128, 8), dtype="fp16", name="decode_23_fp16"),
        # a short prompt: ragged sizes everywhere, biases, GEGLU
        _case("infer", 777, (1472, 704, 48, 4), act="geglu", bias=True, name="prompt_777_geglu_bias"),
        # a prefill chunk of the large layer with skewed expert load
        _case("infer", 4096, (4096, 1024, 128, 8), skew=True, name="prefill_4096_skew"),
        # prefill on fp8 operands with the weights quantised once
        _case("infer", 2048, (4096, 1024, 128, 8), fp8=True, name="prefill_2048_fp8"),
        # the smallest training step of the configurations: launches and host work count
        _case("train", 1024, (512, 256, 8, 2), name="train_1024_small"),
        # an ordinary micro-batch of a mid-sized layer, not a round number of tokens
        _case("train", 6001, (1536, 256, 128, 8), name="train_6001"),
        # narrow layer, many tokens: routing, combine and reductions weigh as much as the GEMMs
        _case("train", 40960, (768, 256, 128, 8), name="train_40960_narrow"),
        # token rounding with the general-routing entry: forward and backward, the router included
        _case("rounding", 16384, (4096, 1024, 256, 8), backward=True, name="rounding_16384"),
        # training on fp8 activation-side operands; the weights change every step, so they are quantised in every one
        _case("train", 8192, (4096, 1024, 128, 8), fp8=True, name="train_8192_fp8"),
        # the headline configuration: the largest step
        _case("train", 32768, (4096, 1024, 128, 8), name="train_32768"),
    ]


def _log_uniform(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case of the same ranges: decode, prefill, training or token rounding; a layer of the configurations or
    one with ragged sizes; any element type, activation, bias, load and operand option that goes with it."""
    largest = _cost(next(c for c in listed() if c["name"] == "train_32768"))
    while True:
        kind = rng.choice(["decode", "decode", "prefill", "prefill", "train", "train", "rounding"])
        fp8 = kind != "rounding" and rng.random() < 0.2
        if rng.random() < 0.3:
            step = 128 if fp8 else 64
            E = rng.choice([8, 16, 32, 48, 64, 128, 256])
            model = (step * rng.randint(512 // step, 4096 // step), step * rng.randint(256 // step, 1536 // step), E,
                     rng.choice([k for k in (1, 2, 4, 6, 8) if k <= E // 4]))
        else:
            model = rng.choice(MODELS)
        if kind == "decode":
            T = _log_uniform(rng, 1, 256)
        elif kind == "prefill":
            T = _log_uniform(rng, 257, 16384)
        elif kind == "train":
            T = _log_uniform(rng, 1000, 40960)
        else:  # enough tokens that rounding to whole tiles leaves the experts their share
            T = rng.randint(max(2048, ROUNDING_TILE * model[2] // model[3]), 32768)
        act, bias = "swiglu", False
        if not fp8 and rng.random() < 0.3:
            act = rng.choice(GATED + UNGATED)
            bias = rng.random() < 0.5
        case = _case({"decode": "infer", "prefill": "infer"}.get(kind, kind), T, model,
                     backward=kind == "train" or (kind == "rounding" and rng.random() < 0.7),
                     dtype="fp16" if rng.random() < 0.25 else "bf16", act=act, bias=bias,
                     skew=kind != "rounding" and rng.random() < 0.3, fp8=fp8)
        if _cost(case) <= largest:
            return case


def _randn(gen, *shape, dtype, std=1.0):
    return torch.empty(*shape, dtype=dtype, device="cuda").normal_(0, std, generator=gen)


def prepare(case, seed):
    """The layer with its weights, the tokens (as they leave a normalisation: unit variance) and, where there is a
    backward pass, the gradient that arrives at the output."""
    T, H, I, E = case["T"], case["H"], case["I"], case["E"]
    dtype, act, backward = DTYPES[case["dtype"]], ActivationType(case["act"]), case["backward"]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    with torch.device("cuda"), torch.no_grad():
        moe = MoE(E, case["K"], H, I, act, case["bias"], 0.02).to(dtype)
        params = [moe.router.weight, moe.c_fc.weight, moe.c_proj.weight]
        for p in params:
            p.normal_(0, 0.02, generator=gen)
        if case["bias"]:
            params += [moe.c_fc.bias, moe.c_proj.bias]
            for p in params[3:]:
                p.normal_(0, 0.01, generator=gen)
        x = _randn(gen, T, H, dtype=dtype)
        if case["skew"]:
            # a direction that all tokens share and every expert's router row answers to by its popularity
            common = torch.full((H,), H ** -0.5)
            rank = torch.randperm(E, generator=gen, device="cuda").float()
            popularity = -2.0 * torch.log(rank + 1.0)
            x.add_(common.to(dtype))
            moe.router.weight.add_((popularity[:, None] * common).to(dtype))
        dout = _randn(gen, T, H, dtype=dtype) if backward else None
    moe.train(backward)
    moe.requires_grad_(backward)
    x.requires_grad_(backward)
    daux = torch.tensor(AUX_COEFFICIENT, device="cuda")
    return dict(case=case, moe=moe, params=params, x=x, dout=dout, daux=daux)


def run(state):
    case = state["case"]
    with ExitStack() as scope:
        if case["fp8"]:
            scope.enter_context(enable_fp8_forward())
            if case["backward"]:
                scope.enter_context(enable_fp8_backward())
                scope.enter_context(cache_quantized_weights(False))
        return (_run_rounding if case["task"] == "rounding" else _run_module)(state)


def _run_module(state):
    moe, x = state["moe"], state["x"]
    if not state["case"]["backward"]:
        with torch.no_grad():
            return moe(x)
    out, aux = moe(x)
    grads = torch.autograd.grad([out, aux], [x] + state["params"], grad_outputs=[state["dout"], state["daux"]])
    return [out.detach(), aux.detach(), *grads]


def _run_rounding(state):
    case, moe, x = state["case"], state["moe"], state["x"]
    with torch.no_grad():
        logits = F.linear(x, moe.router.weight)
        scores, tokens, experts = token_choice_rounding(logits, case["K"], ROUNDING_TILE, "nr")
    scores = scores.float().requires_grad_(case["backward"])
    with torch.set_grad_enabled(case["backward"]):
        out, frequency = moe_general_routing_inputs(
            x, scores, tokens, experts, moe.c_fc.weight.permute(1, 2, 0), moe.c_fc.bias, moe.c_proj.weight.permute(1, 2, 0),
            moe.c_proj.bias, case["E"], torch.cuda.current_stream().cuda_stream, moe.activation_function,
            not case["backward"])
    if not case["backward"]:
        return [out, frequency]
    dx, dscores, *grads = torch.autograd.grad(out, [x, scores] + state["params"][1:], grad_outputs=state["dout"])
    dprobabilities = torch.zeros(case["T"], case["E"], device="cuda")  # what the router's softmax gets back
    dprobabilities[tokens, experts] = dscores
    return [out.detach(), frequency, dx, dprobabilities, *grads]


def _pick_probabilities(case):
    """The probability that a token picks an expert, by the expert's popularity rank."""
    H, E, K = case["H"], case["E"], case["K"]
    if not case["skew"]:
        return [K / E] * E
    spread = 0.02 * H ** 0.5 * 2 ** 0.5  # of a logit around the expert's popularity
    lo, hi = -100.0, 100.0
    for _ in range(60):  # the threshold that K experts pass on average
        mid = (lo + hi) / 2
        p = [0.5 * math.erfc((mid + 2.0 * math.log(r + 1.0)) / spread) for r in range(E)]
        lo, hi = (mid, hi) if sum(p) > K else (lo, mid)
    return p


def work(case):
    """Bytes: the tokens, the weights of the experts that are picked, and with a backward pass the output gradient, each
    read once; the output and the gradients written once.  Operations: the expert GEMMs and the router's."""
    T, H, I, E, K = case["T"], case["H"], case["I"], case["E"], case["K"]
    expert = (3 if is_glu(ActivationType(case["act"])) else 2) * I * H  # weights of one expert
    touched = sum(1.0 - (1.0 - q) ** T for q in _pick_probabilities(case))
    byte = 1 if case["fp8"] and not case["backward"] else 2  # a server quantises its weights once
    passes = 3 if case["backward"] else 1
    flops = passes * 2.0 * T * (K * expert + H * E)
    if not case["backward"]:
        return {"bytes": touched * expert * byte + E * H * 2 + 2 * T * H * 2, "flops": flops}
    return {"bytes": (touched + E) * expert * 2 + 2 * E * H * 2 + 4 * T * H * 2, "flops": flops}


def _cost(case):
    w = work(case)
    return w["flops"] / 2.5e15 + w["bytes"] / 8e12


def tolerance(case):
    """Four times the distance of outputs and gradients from the same layer evaluated in fp32 with the same routing:
    bf16 2.9e-3 to 6.8e-3 over sizes, activations and loads, fp16 2.9e-4 to 7.2e-4 (the rounding of the stored
    tensors).  On fp8 operands a different summation order also moves values across a quantisation boundary."""
    return {"rel": 3e-3 if case["dtype"] == "fp16" and not case["fp8"] else 2e-2}
