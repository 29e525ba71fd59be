"""The work that a user of the package has it do, as cases that can be timed.

A case is one ``FMoETransformerMLP`` layer over one batch of tokens: a forward without gradients
(``"mode": "infer"``: decoding steps of a few tokens, prompts of some thousand) or one training step
(``"train"``: forward and backward, gradients of the input, the gate and the experts).  The sizes are the
layer's own defaults, those of the benchmark's configurations and generic ones between them.

Fields of a case: ``mode``; ``tokens``, ``d_model``, ``d_hidden``, ``experts``, ``top_k``; ``dtype`` ("bf16", "f16",
"f32"); ``act`` ("gelu", "relu"); ``fused`` (the chunked pipeline instead of the module path); ``routing``, how the gate
spreads the tokens: "even" (a freshly initialised gate), "skewed" (per-expert biases of the size of the
logits' spread), "zipf" (a few experts take most tokens), "capacity" (even, and every expert keeps at most
1.2 times its share, the rest of its slots are dropped).
"""
import math

import torch

import fastermoe_amd as fmoe
from fastermoe_amd.gates import NaiveGate
from fastermoe_amd.gates.utils import limit_by_capacity

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


class CapacityGate(NaiveGate):
    """Top-k with at most 1.2 times an even share of the slots per expert."""

    def forward(self, inp):
        idx, score = super().forward(inp)
        cap = math.ceil(1.2 * idx.numel() / self.num_expert)
        return limit_by_capacity(idx, self.num_expert, self.world_size, cap)[2], score


def _case(name, mode, tokens, d_model, d_hidden, experts, top_k, dtype, routing="even", act="gelu", fused=False):
    case = {"mode": mode, "tokens": tokens, "d_model": d_model, "d_hidden": d_hidden, "experts": experts,
            "top_k": top_k, "dtype": dtype, "routing": routing, "act": act, "fused": fused}
    return dict(case, name=name) if name else case


def listed():
    return [
        # one token of a text being generated, through a layer of the default size
        _case("decode-1-default-layer", "infer", 1, 1024, 4096, 32, 2, "bf16"),
        # a decoding step of 32 sequences through few large experts: streams every weight once
        _case("decode-32-large-experts", "infer", 32, 4096, 14336, 8, 2, "bf16"),
        # a decoding step of 64 sequences through many small experts, a row or two each
        _case("decode-64-many-experts", "infer", 64, 2048, 1024, 256, 8, "bf16", "skewed"),
        # one short prompt of odd length, top-1 of 64 experts with skewed use
        _case("prompt-509-top1", "infer", 509, 2048, 8192, 64, 1, "f16", "zipf"),
        # a batch of prompts through the large experts
        _case("prompt-4096-large-experts", "infer", 4096, 4096, 14336, 8, 2, "bf16"),
        # a small training step of ragged size, with ReLU experts
        _case("train-1000-relu", "train", 1000, 768, 3072, 16, 2, "f16", "even", "relu"),
        # feature sizes that are no multiple of the vector width
        _case("train-777-odd-features", "train", 777, 500, 1302, 12, 2, "bf16"),
        # the benchmark's five training steps
        _case("train-4096-f32", "train", 4096, 512, 1024, 8, 2, "f32"),
        _case("train-16384-capacity", "train", 16384, 1024, 4096, 16, 2, "bf16", "capacity"),
        _case("train-16384-top1-zipf", "train", 16384, 2048, 8192, 64, 1, "bf16", "zipf"),
        _case("train-32768-fused", "train", 32768, 4096, 14336, 8, 2, "bf16", "even", "gelu", True),
        _case("train-8192-many-experts", "train", 8192, 2048, 1024, 256, 8, "bf16", "skewed"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# the most a drawn case may cost: flop of a step per element type (the largest listed step is 4.6e13 in bf16),
# the same where the feature sizes are odd, and bytes of the experts' weights (the largest listed layer is 4.3e9)
MAX_FLOPS = {"bf16": 3e13, "f16": 3e13, "f32": 1e12}
MAX_FLOPS_ODD = 2e11
MAX_WEIGHT_BYTES = 4.2e9


def draw(rng):
    while True:
        mode = rng.choice(["decode", "prompt", "train", "train"])
        tokens = {"decode": lambda: _log_int(rng, 1, 256), "prompt": lambda: _log_int(rng, 256, 8192),
                  "train": lambda: _log_int(rng, 512, 32768)}[mode]()
        if tokens > 64 and rng.random() < 0.5:
            tokens = max(64, tokens // 64 * 64)   # batches of whole sequences as often as odd numbers of tokens
        d_model = 64 * _log_int(rng, 8, 64)
        d_hidden = 64 * max(8, int(d_model / 64 * rng.choice([0.5, 1, 2, 3.5, 4])))
        experts = rng.choice([4, 8, 8, 12, 16, 32, 64, 128, 256])
        top_k = rng.choice([1, 2, 2, 4] + ([8] if experts >= 32 else []))
        dtype = rng.choice(["bf16", "bf16", "bf16", "f16", "f32"])
        odd = rng.random() < 0.1
        if odd:
            d_model, d_hidden = d_model - rng.randrange(1, 60), d_hidden - rng.randrange(1, 60)
        case = _case("", "train" if mode == "train" else "infer", tokens, d_model, d_hidden, experts, top_k, dtype,
                     rng.choice(["even", "even", "skewed", "capacity"] + (["zipf"] if experts >= 16 else [])),
                     rng.choice(["gelu", "gelu", "relu"]),
                     mode == "train" and not odd and rng.random() < 0.2)
        flops = (12 if mode == "train" else 4) * tokens * top_k * d_model * d_hidden
        if (flops <= (MAX_FLOPS_ODD if odd else MAX_FLOPS[dtype])
                and 2 * experts * d_model * d_hidden * DTYPES[dtype].itemsize <= MAX_WEIGHT_BYTES):
            return case


def prepare(case, seed):
    dev = torch.device("cuda")
    dtype = DTYPES[case["dtype"]]
    gen = torch.Generator(device=dev).manual_seed(seed)
    d, h, e = case["d_model"], case["d_hidden"], case["experts"]
    with dev:
        layer = fmoe.FMoETransformerMLP(
            num_expert=e, d_model=d, d_hidden=h, top_k=case["top_k"],
            gate=CapacityGate if case["routing"] == "capacity" else NaiveGate,
            activation=torch.nn.GELU() if case["act"] == "gelu" else torch.nn.ReLU())
    layer = layer.to(dtype)
    layer.enable_fuse = case["fused"]
    with torch.no_grad():
        # unit-variance activations all the way, as a trained layer between normalisations has
        for lin, fan_in in ((layer.experts.htoh4, d), (layer.experts.h4toh, h)):
            bound = math.sqrt(3.0 / fan_in)
            lin.weight.uniform_(-bound, bound, generator=gen)
            lin.bias.normal_(0.0, 0.1, generator=gen)
        gate = layer.gate.gate
        bound = math.sqrt(3.0 / d)   # logits ~ N(0, 1)
        gate.weight.uniform_(-bound, bound, generator=gen)
        if case["routing"] == "skewed":
            gate.bias.normal_(0.0, 0.5, generator=gen)
        elif case["routing"] == "zipf":
            share = torch.arange(1, e + 1, device=dev, dtype=torch.float32) ** -1.2
            share = share[torch.randperm(e, device=dev, generator=gen)]
            gate.bias.copy_(0.78 * torch.log(share / share.sum()))   # (0.78: normal noise in a Gumbel's place)
        else:
            gate.bias.normal_(0.0, 0.02, generator=gen)
    x = torch.randn(case["tokens"], d, device=dev, generator=gen).to(dtype)
    state = {"layer": layer, "x": x, "grad": None}
    if case["mode"] == "train":
        layer.train()
        x.requires_grad_(True)
        state["grad"] = torch.randn(case["tokens"], d, device=dev, generator=gen).to(dtype)
    else:
        layer.eval()
    return state


def run(state):
    layer, x = state["layer"], state["x"]
    if state["grad"] is None:
        with torch.no_grad():
            return layer(x)
    layer.zero_grad(set_to_none=True)
    x.grad = None
    out = layer(x)
    out.backward(state["grad"])
    grads = {name: p.grad for name, p in layer.named_parameters()}
    return dict(grads, out=out.detach(), grad_x=x.grad)


def work(case):
    n, d, h, e, k = (case[f] for f in ("tokens", "d_model", "d_hidden", "experts", "top_k"))
    size = DTYPES[case["dtype"]].itemsize
    train = case["mode"] == "train"
    # experts that some slot names, on logits of the gate's distribution: the weights that have to be read
    # (a training step writes every expert's gradient)
    gen = torch.Generator().manual_seed(0)
    bias = torch.zeros(e)
    if case["routing"] == "skewed":
        bias = 0.5 * torch.randn(e, generator=gen)
    elif case["routing"] == "zipf":
        bias = -0.78 * 1.2 * torch.log(torch.arange(1, e + 1, dtype=torch.float32))
    named = (torch.randn(n, e, generator=gen) + bias).topk(k, dim=1).indices.unique().numel()
    expert = 2 * d * h + d + h
    rows, weights = 2 * n * d, named * expert + e * (d + 1)
    if train:
        rows, weights = 2 * rows, weights + e * (expert + d + 1)
    return {"bytes": size * (rows + weights), "flops": (3 if train else 1) * (4 * n * k * d * h + 2 * n * d * e)}


def tolerance(case):
    # about four times what the listed and some drawn cases differ by from the same path in float64
    # (bf16: rel 3.4e-3, max 0.068 in a weight gradient over a few rows; f16: an eighth; f32: rel 1.3e-6)
    if case["dtype"] == "f32":
        return {"rel": 5e-6, "max": 1.5e-4}
    if case["dtype"] == "f16":
        return {"rel": 1.7e-3, "max": 0.035}
    return {"rel": 0.014, "max": 0.27}
