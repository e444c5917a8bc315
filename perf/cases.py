"""The calls whose speed this framework is judged by: its linears and its MoE blocks, through the entry points a model's
code calls, from one decoded token to a prefill chunk.

Every case is a dict of plain values whose "path" names the entry point:

  linear   one projection: "w3" (three-bit) and "w3_two_bit" through `w3.w3_linear` (at most 128 rows, the size its
           decode copies serve), "nvfp4" through `ops.nvfp4_linear` (any number of rows)
  mlp      the dense SwiGLU block `Mlp`: three-bit copies (its down projection then takes E4M3 activations) or NVFP4
  moe      `MoeLayer` on three-bit experts with the shared expert and its gate: router product, top-k, experts, combine;
           "requests" > 0: a decode or verify forward of a graph padded to that many requests (the last of them holds
           none) of rows / requests tokens each; "budget" > 0: its budgeted expert selection
  latent   `NemotronMoe` on NVFP4 experts: router and latent projections, sigmoid top-k, experts, combine, projection
           back; "shared" > 0: with a shared expert of that intermediate size

`listed` holds one of each in the sizes of the benchmark configurations (README and bench.py name them) and `draw` other
sizes of the same ranges, ragged ones among them.
"""
from __future__ import annotations

import math
from types import SimpleNamespace

import torch

from hibana_amd import synthetic
from hibana_amd.kernels import ops, w3
from hibana_amd.model.flashnext_moe import MoeLayer
from hibana_amd.model.mlp import Mlp
from hibana_amd.model.nemotron_moe import NemotronMoe

KEEP, PER_REQUEST = 4, 12  # budgeted selection: a token's own experts, distinct experts a request
NOISE = 1.28  # standard deviation of the logits around their expert's popularity (a Gumbel variable's)
MOST_FLOPS = 5.3e11  # of a drawn case: the largest listed one's
LEAN = 16.0   # how far the activations lean towards the direction that carries the popularity


def listed() -> list[dict]:
    return [
        # one token through an attention-sized projection: the smallest call, launch and latency
        {"name": "w3_linear_1", "path": "linear", "format": "w3", "rows": 1, "out": 5120, "in": 5120},
        # a draft model's vocabulary head on its two-bit copy, a few drafted tokens
        {"name": "draft_head_12", "path": "linear", "format": "w3_two_bit", "rows": 12, "out": 51200, "in": 2048},
        # an MLP up-projection in NVFP4: eight sequences decoding, a ragged verify batch, a whole prefill chunk (the largest)
        {"name": "nvfp4_linear_8", "path": "linear", "format": "nvfp4", "rows": 8, "out": 25600, "in": 5120},
        {"name": "nvfp4_linear_77", "path": "linear", "format": "nvfp4", "rows": 77, "out": 25600, "in": 5120},
        {"name": "nvfp4_linear_2048", "path": "linear", "format": "nvfp4", "rows": 2048, "out": 25600, "in": 5120},
        # the dense block of a decode step of four sequences on its three-bit copies
        {"name": "mlp_w3_4", "path": "mlp", "format": "w3", "rows": 4, "hidden": 5120, "inter": 25600},
        # the routed layer: one token; four sequences verifying eight drafted tokens each with skewed routing; five
        # slots of a padded graph under a budget of experts; a ragged prefill chunk
        {"name": "moe_decode_1", "path": "moe", "rows": 1, "hidden": 2048, "inter": 512, "experts": 512, "topk": 10, "zipf": 0.0, "requests": 0, "budget": 0},
        {"name": "moe_verify_32", "path": "moe", "rows": 32, "hidden": 2048, "inter": 512, "experts": 512, "topk": 10, "zipf": 1.1, "requests": 0, "budget": 0},
        {"name": "moe_budget_40", "path": "moe", "rows": 40, "hidden": 2048, "inter": 512, "experts": 512, "topk": 10, "zipf": 1.1, "requests": 5, "budget": 64},
        {"name": "moe_prefill_1543", "path": "moe", "rows": 1543, "hidden": 2048, "inter": 512, "experts": 512, "topk": 10, "zipf": 1.1, "requests": 0, "budget": 0},
        # the latent block: four sequences decoding, a prefill chunk
        {"name": "latent_decode_4", "path": "latent", "rows": 4, "hidden": 4096, "latent": 1024, "inter": 2688, "experts": 512, "topk": 22, "shared": 5376},
        {"name": "latent_prefill_2048", "path": "latent", "rows": 2048, "hidden": 4096, "latent": 1024, "inter": 2688, "experts": 512, "topk": 22, "shared": 0},
    ]


def _between(rng, low: float, high: float, step: int = 1) -> int:
    """A multiple of `step` between the two, spread evenly over the logarithm."""
    value = math.exp(rng.uniform(math.log(low), math.log(high)))
    return max(step, int(round(value / step)) * step)


def draw(rng) -> dict:
    path = rng.choice(["linear", "linear", "linear", "mlp", "moe", "moe", "moe", "latent", "latent"])
    if path == "linear":
        form = rng.choice(["w3", "w3_two_bit", "nvfp4", "nvfp4"])
        case = {"path": path, "format": form, "rows": _between(rng, 1, 2048 if form == "nvfp4" else 128),
                "out": _between(rng, 1024, 25600 if form == "nvfp4" else 51200, 64 if form == "nvfp4" else 128), "in": _between(rng, 512, 5120, 128)}
    elif path == "mlp":
        form = rng.choice(["w3", "nvfp4"])
        case = {"path": path, "format": form, "rows": _between(rng, 1, 128 if form == "w3" else 512), "hidden": _between(rng, 1024, 5120, 128),
                "inter": _between(rng, 1024, 12800, 128)}
    elif path == "moe":
        rows, requests, budget = _between(rng, 1, 2048), 0, 0
        if rng.random() < 0.4:  # a padded decode (one token a request) or verify forward
            steps = rng.choice([1, 3, 8])
            requests = _between(rng, 2, 16)
            rows, budget = requests * steps, rng.choice([0, 64])
        case = {"path": path, "rows": rows, "hidden": _between(rng, 1024, 2560, 128), "inter": _between(rng, 256, 768, 128), "experts": _between(rng, 64, 512, 8),
                "topk": rng.randint(6, 12), "zipf": rng.choice([0.0, 1.1]), "requests": requests, "budget": budget}
    else:
        case = {"path": path, "rows": _between(rng, 1, 2048), "hidden": _between(rng, 2048, 4096, 128), "latent": _between(rng, 512, 1024, 128),
                "inter": _between(rng, 1024, 2688, 128), "experts": _between(rng, 128, 512, 8), "topk": rng.randint(8, 22),
                "shared": rng.choice([0, _between(rng, 2048, 5376, 128)])}
        while work(case)["flops"] > MOST_FLOPS:
            case["rows"] = case["rows"] * 3 // 4
    return case


def _logits_router(experts: int, hidden: int, zipf: float, g, device):
    """BF16 router weights and the FP32 direction its inputs lean along: a row's logits are the log popularity of the
    experts (Zipf over a random order; none for `zipf` 0) plus noise."""
    direction = torch.nn.functional.normalize(torch.randn(hidden, device=device, generator=g), dim=0)
    rank = torch.randperm(experts, device=device, generator=g).float() + 1.0
    logp = -zipf * rank.log()
    noise = torch.randn(experts, hidden, device=device, generator=g) * ((NOISE if zipf else 1.0) / hidden ** 0.5)
    return (noise + (logp - logp.mean())[:, None] / LEAN * direction).bfloat16(), direction * (LEAN if zipf else 0.0)


def _w3_linear(out: int, k: int, seed: int, codebook: str = "lloyd"):
    return w3.tile(synthetic.w3_matrix(out, k, seed, codebook=codebook), release=True)


def prepare(case: dict, seed: int) -> SimpleNamespace:
    device = torch.device("cuda")
    g = torch.Generator(device=device).manual_seed(seed + 1)
    state = SimpleNamespace(path=case["path"], ctx=None)
    rows = case["rows"]
    seed *= 16  # the weights' own seeds
    if state.path == "linear":
        state.format = case["format"]
        if state.format == "nvfp4":
            state.weight = synthetic.nvfp4_linear(case["out"], case["in"], seed)
        else:
            state.weight = _w3_linear(case["out"], case["in"], seed, "lloyd" if state.format == "w3" else "lloyd2")
        state.x = torch.randn(rows, case["in"], device=device, generator=g).bfloat16()
    elif state.path == "mlp":
        hidden, inter = case["hidden"], case["inter"]
        # weights of a trained block's size: an output of the order of one (the random codes have a spread of about 3)
        gate_up = synthetic.nvfp4_linear(2 * inter, hidden, seed, global_scale=0.3 / hidden ** 0.5)
        down = synthetic.nvfp4_linear(hidden, inter, seed + 1, global_scale=0.3 / inter ** 0.5)
        if case["format"] == "w3":  # serve it from the three-bit copies, as HIBANA_W3_DECODE=1 does
            gate_up.w3, down.w3 = _w3_linear(2 * inter, hidden, seed + 2), _w3_linear(hidden, inter, seed + 3)
            w3.set_enabled(True)
        state.block = Mlp(gate_up, down)
        state.x = torch.randn(rows, hidden, device=device, generator=g).bfloat16()
    elif state.path == "moe":
        hidden, inter, experts = case["hidden"], case["inter"], case["experts"]
        router, lean = _logits_router(experts, hidden, case["zipf"], g, device)
        gate = torch.randn(1, hidden, device=device, generator=g) / hidden ** 0.5
        state.block = MoeLayer(router, gate, synthetic.w3_experts(experts, hidden, inter, True, seed), case["topk"],
                               shared=synthetic.w3_experts(1, hidden, inter, True, seed + 1), keep=KEEP if case["budget"] else 0,
                               budget=case["budget"], per_request=PER_REQUEST if case["budget"] else 0)
        state.x = (torch.randn(rows, hidden, device=device, generator=g) + lean).bfloat16()
        if case["requests"]:
            slots = torch.arange(1, case["requests"] + 1, device=device, dtype=torch.int32)
            slots[-1] = 0  # the graph's last request is padding
            steps = rows // case["requests"]
            state.ctx = SimpleNamespace(mode="decode", slots=slots) if steps == 1 else SimpleNamespace(mode="verify", seq_slots=slots, verify_steps=steps)
    else:
        hidden, latent, inter, experts = case["hidden"], case["latent"], case["inter"], case["experts"]
        router, _ = _logits_router(experts, hidden, 0.0, g, device)
        fc1 = (torch.randn(latent, hidden, device=device, generator=g) / hidden ** 0.5).bfloat16()
        fc2 = (torch.randn(hidden, latent, device=device, generator=g) / latent ** 0.5).bfloat16()
        bias = torch.rand(experts, device=device, generator=g) * 0.1
        up = down = None
        if case["shared"]:
            up = synthetic.nvfp4_linear(case["shared"], hidden, seed + 1)
            down = synthetic.nvfp4_linear(hidden, case["shared"], seed + 2)
        state.block = NemotronMoe(torch.cat([router, fc1]), bias, fc2, synthetic.nvfp4_experts(experts, latent, inter, seed), case["topk"],
                                  shared_up=up, shared_down=down)
        state.x = torch.randn(rows, hidden, device=device, generator=g).bfloat16()
    return state


def run(state: SimpleNamespace) -> torch.Tensor:
    if state.path == "linear":
        return ops.nvfp4_linear(state.x, state.weight) if state.format == "nvfp4" else w3.w3_linear(state.x, state.weight)
    if state.path == "mlp":
        return state.block(state.x)
    return state.block(state.x, state.ctx)


def _w3_bytes(n: int, k: int, bits: int = 3) -> float:
    return n * k * bits / 8 + n * k / 32 + 4 * n


def _nvfp4_bytes(n: int, k: int) -> float:
    return n * k / 2 + n * k / 16


def _distinct(rows: int, experts: int, topk: int, zipf: float) -> float:
    """The experts that `rows` draws of `topk` name, on average: an expert is in a row's top k with a probability q
    that grows with its popularity, the q adding up to topk."""
    p = [(e + 1.0) ** -zipf for e in range(experts)]
    low, high = 0.0, 1e9
    for _ in range(100):
        mid = math.sqrt(low * high) if low else high / 2
        if sum(1.0 - math.exp(-mid * v) for v in p) < topk:
            low = mid
        else:
            high = mid
        if low and high / low < 1.0001:
            break
    return sum(1.0 - math.exp(-high * v * rows) for v in p)


def work(case: dict) -> dict:
    """Weights that a call names once (in the checkpoint's formats), activations in and out once; the products of its
    real rows."""
    rows = case["rows"]
    if case["path"] == "linear":
        n, k = case["out"], case["in"]
        weights = _nvfp4_bytes(n, k) if case["format"] == "nvfp4" else _w3_bytes(n, k, 3 if case["format"] == "w3" else 2)
        return {"bytes": weights + 2.0 * rows * (n + k), "flops": 2.0 * rows * n * k}
    if case["path"] == "mlp":
        h, i = case["hidden"], case["inter"]
        size = _w3_bytes if case["format"] == "w3" else _nvfp4_bytes
        return {"bytes": size(2 * i, h) + size(h, i) + 4.0 * rows * h, "flops": 6.0 * rows * h * i}
    experts, topk = case["experts"], case["topk"]
    if case["path"] == "moe":
        h, i = case["hidden"], case["inter"]
        real = rows - rows // case["requests"] if case["requests"] else rows
        distinct = _distinct(real, experts, topk, case["zipf"])
        if case["budget"]:
            distinct = min(distinct, min(case["budget"], max(MoeLayer.MIN_CAP, PER_REQUEST * (case["requests"] - 1))))
        one = _w3_bytes(2 * i, h) + _w3_bytes(h, i)
        return {"bytes": (distinct + 1.0) * one + 2.0 * experts * h + 4.0 * rows * h,
                "flops": 2.0 * rows * experts * h + 6.0 * h * i * (real * topk + rows)}
    h, latent, i, shared = case["hidden"], case["latent"], case["inter"], case["shared"]
    distinct = _distinct(rows, experts, topk, 0.0)
    return {"bytes": distinct * 2 * _nvfp4_bytes(i, latent) + 2 * _nvfp4_bytes(shared, h) + 2.0 * (experts + 2 * latent) * h + 4.0 * rows * h,
            "flops": 2.0 * rows * h * (experts + 2 * latent) + 4.0 * rows * topk * i * latent + 4.0 * rows * shared * h}


def tolerance(case: dict) -> dict:
    """BF16 results of FP32 sums, with a BF16 rounding or two on the way."""
    return {"rel": 1e-2}
