"""The engine's performance cases: the calls that a serving node makes, by size.

listed() holds fixed cases, draw() more of the same ranges; prepare() builds
what a program keeps between calls (resident experts, layer, router weights)
and its activations from a seed; run() is one call through the public entry
points of constellation_amd.engine; exact() restates it in 64-bit torch.

Every case is the DeepSeek-V3 MoE geometry that bench.py measures: hidden
7168, inter 2048, 256 experts in 8 groups, top 4 groups, top 8 experts, fp8
weights with 128 x 128 block scales, one shared expert.  Kinds:
  route    the router alone (the server asks for routes, experts live elsewhere)
  layer    router + routed experts + shared expert, all experts on this GPU
  share    routes given, this GPU holding one expert in four (one node of four)
  expert   one expert over a batch on the device
  host     one expert, host bytes in and out (the wire's InferRequest)
  request  a whole layer, host bytes in and out (MoeLayerRequest)
"""
import math

import numpy as np
import torch

from constellation_amd import moe_layer_protocol as wire
from constellation_amd._lib import FP16
from constellation_amd.engine import LAYOUT_TILE16, Context, Expert, Layer

HIDDEN, INTER, EXPERTS, GROUPS, TOP_GROUPS, TOP_K, SCALE = 7168, 2048, 256, 8, 4, 8, 2.5
BLOCK = 128
EXPERT_BYTES = 3 * HIDDEN * INTER + 3 * (HIDDEN // BLOCK) * (INTER // BLOCK) * 4
EXPERT_FLOPS = 6 * HIDDEN * INTER  # per token and expert
ROUTER_BYTES = EXPERTS * HIDDEN * 2 + EXPERTS * 4
LARGEST = 4096  # tokens of one call


def listed():
    return [
        # the routing decision for one new token: launches and latency only
        {"name": "route_1", "kind": "route", "tokens": 1, "zipf": 0.0},
        # decode of one sequence: the headline call, bound by 400 MB of weights
        {"name": "layer_1", "kind": "layer", "tokens": 1, "zipf": 0.0},
        # decode of a handful of sequences
        {"name": "layer_6", "kind": "layer", "tokens": 6, "zipf": 0.0},
        # a full decode batch
        {"name": "layer_16", "kind": "layer", "tokens": 16, "zipf": 0.0},
        # one node of four serving a decode batch with hot experts
        {"name": "share_32", "kind": "share", "tokens": 32, "zipf": 0.25},
        # a short prompt's prefill chunk, hot experts
        {"name": "layer_512", "kind": "layer", "tokens": 512, "zipf": 0.25},
        # a ragged, longer prompt: weights and matrix work are of one size
        {"name": "layer_1511", "kind": "layer", "tokens": 1511, "zipf": 0.0},
        # the largest chunk: over a hundred tokens per expert
        {"name": "layer_4096", "kind": "layer", "tokens": LARGEST, "zipf": 0.0},
        # the reference's wire request: one expert, one token, fp16 host bytes
        {"name": "host_1", "kind": "host", "tokens": 1, "dtype": "fp16"},
        # one expert over a decode batch
        {"name": "expert_13", "kind": "expert", "tokens": 13, "dtype": "bf16"},
        # one expert (the shared one, say) over a prefill chunk
        {"name": "expert_300", "kind": "expert", "tokens": 300, "dtype": "fp16"},
        # one message per layer from the server: routes and activations as host bytes
        {"name": "request_5", "kind": "request", "tokens": 5, "zipf": 0.0},
    ]


def draw(rng):
    kind = rng.choice(["layer", "layer", "layer", "share", "share", "expert", "expert", "expert",
                       "host", "request", "route"])
    most = {"layer": LARGEST, "share": 2048, "expert": LARGEST, "host": 64, "request": 256,
            "route": LARGEST}[kind]
    case = {"kind": kind, "tokens": min(most, int(round(math.exp(rng.uniform(0.0, math.log(most + 0.49))))))}
    if kind in ("expert", "host"):
        case["dtype"] = "fp16" if kind == "host" else rng.choice(["bf16", "fp16"])
    else:
        case["zipf"] = rng.choice([0.0, round(rng.uniform(0.02, 0.25), 3)])
    return case


class State:
    """What the program keeps; the experts go back to the arena with it."""

    def __init__(self):
        self.ctx, self.layer, self.experts = Context(0), None, []

    def __del__(self):
        if self.layer is not None:
            self.layer.close()
        for e in self.experts:
            e.free()
        self.ctx.close()


def _resident(case):
    return range(0, EXPERTS, 4) if case["kind"] == "share" else range(EXPERTS)


def _dtype(case):
    return torch.float16 if case.get("dtype") == "fp16" or case["kind"] == "request" else torch.bfloat16


def prepare(case, seed):
    s = State()
    s.case = dict(case)
    kind, n = case["kind"], case["tokens"]
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape, std, dtype):
        return (torch.randn(*shape, generator=gen, device="cuda") * std).to(dtype)

    s.x = normal(n, HIDDEN, std=1.0, dtype=_dtype(case))
    base = 4 * (EXPERTS + 1) * (seed % 4096)

    def expert(e):
        s.experts.append(Expert.generate(0, seed, base + 4 * e, HIDDEN, INTER, BLOCK, 0.02))
        return s.experts[-1]

    if kind in ("expert", "host"):
        s.expert = expert(0)
        s.x_bytes = s.x.cpu().numpy().tobytes() if kind == "host" else None
        return s
    s.w_router = normal(EXPERTS, HIDDEN, std=0.02, dtype=torch.bfloat16)
    rank = torch.randperm(EXPERTS, generator=gen, device="cuda") + 1
    s.bias = normal(EXPERTS, std=0.01, dtype=torch.float32) + case["zipf"] * rank.float() ** -1.1
    if kind == "route":
        return s
    held = set(_resident(case))
    s.mask = None
    if len(held) < EXPERTS:
        s.mask = torch.tensor([e in held for e in range(EXPERTS)], dtype=torch.uint8, device="cuda")
    local = [expert(e) if e in held else None for e in range(EXPERTS)]
    shared = None if kind == "share" else expert(EXPERTS)
    s.layer = Layer(s.ctx, local, shared)
    if kind != "layer":
        # routes as the server sends them
        s.ids, s.w = s.ctx.route(s.x.to(torch.bfloat16), s.w_router, s.bias, resident=s.mask, n_group=GROUPS,
                                 topk_group=TOP_GROUPS, top_k=TOP_K, routed_scaling_factor=SCALE)
    if kind == "request":
        s.body = wire.encode_moe_layer_request({
            "layer_id": 3, "batch_size": n, "hidden_dim": HIDDEN, "top_k": TOP_K, "input_dtype": FP16,
            "output_dtype": FP16, "flags": wire.FLAG_SHARED, "expert_ids": s.ids.cpu().numpy(),
            "expert_weights": s.w.cpu().numpy(), "activation": s.x.cpu().numpy().tobytes()})
    torch.cuda.synchronize()
    return s


def run(s):
    kind, n = s.case["kind"], s.case["tokens"]
    options = dict(n_group=GROUPS, topk_group=TOP_GROUPS, top_k=TOP_K, routed_scaling_factor=SCALE)
    if kind == "route":
        return s.ctx.route(s.x, s.w_router, s.bias, **options)
    if kind == "layer":
        y, _, ids, w = s.ctx.moe_layer(s.layer, s.x, s.w_router, s.bias, **options)
        return y, ids, w
    if kind == "share":
        return s.ctx.moe(s.layer, s.x, s.ids, s.w)
    if kind == "expert":
        return s.ctx.expert_run(s.expert, s.x)
    if kind == "host":
        return np.frombuffer(s.ctx.expert_run_host(s.expert, s.x_bytes, FP16, n, FP16), np.float16).reshape(n, HIDDEN)
    body = s.ctx.moe_layer_request(s.layer, s.body)
    return np.frombuffer(body, np.float16, offset=len(body) - 2 * n * HIDDEN).reshape(n, HIDDEN)


def work(case):
    kind, n = case["kind"], case["tokens"]
    act = 2 * n * HIDDEN * 2  # activations in and out
    if kind == "route":
        return {"bytes": ROUTER_BYTES + act // 2 + n * TOP_K * 8, "flops": 2 * n * EXPERTS * HIDDEN}
    if kind in ("expert", "host"):
        return {"bytes": EXPERT_BYTES + act, "flops": n * EXPERT_FLOPS}
    held = len(_resident(case))
    hit = held * (1.0 - (1.0 - TOP_K / held) ** n)  # distinct experts, even routing
    out = {"bytes": hit * EXPERT_BYTES + act + n * TOP_K * 8, "flops": n * TOP_K * EXPERT_FLOPS}
    if kind != "share":
        out["bytes"] += EXPERT_BYTES
        out["flops"] += n * EXPERT_FLOPS
    if kind == "layer":
        out["bytes"] += ROUTER_BYTES
        out["flops"] += 2 * n * EXPERTS * HIDDEN
    return out


def tolerance(case):
    if case["kind"] == "route":
        return {"rel": 1.2e-7, "max": 2.4e-7}  # weights: one rounding to 32 bits of a 64-bit value
    if _dtype(case) == torch.float16:
        return {"rel": 8e-4, "max": 2e-3}  # four times one rounding to 11 bits (2.1e-4, 4.9e-4)
    return {"rel": 6.5e-3, "max": 1.6e-2}  # four times one rounding to 8 bits (1.7e-3, 3.9e-3)


# ---- the same in 64 bits ---------------------------------------------------

class _Memory:
    """Device memory of an expert as a tensor."""

    def __init__(self, ptr, shape, kind):
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": kind, "version": 2}


def _matrix(ptr, scales, rows, cols, tiled):
    q = torch.as_tensor(_Memory(ptr, (rows * cols,), "|u1"), device="cuda").clone()
    if tiled:  # tiles of 16 rows x 128 columns: [row group][column block][quarter][row][32]
        q = q.view(rows // 16, cols // BLOCK, 4, 16, 32).permute(0, 3, 1, 2, 4)
    v = q.reshape(rows, cols).view(torch.float8_e4m3fn).to(torch.float32).to(torch.float64)
    g = torch.as_tensor(_Memory(scales, (rows // BLOCK, cols // BLOCK), "<f4"), device="cuda").to(torch.float64)
    return v * g.repeat_interleave(BLOCK, 0).repeat_interleave(BLOCK, 1)


def _mlp(e, x):
    d = e.desc
    tiled = d.gu_layout == LAYOUT_TILE16
    gate = x @ _matrix(d.w_gate, d.s_gate, INTER, HIDDEN, tiled).T
    up = x @ _matrix(d.w_up, d.s_up, INTER, HIDDEN, tiled).T
    return (gate * torch.sigmoid(gate) * up) @ _matrix(d.w_down, d.s_down, HIDDEN, INTER, False).T


def _routes(s):
    score = torch.sigmoid(s.x.to(torch.float64) @ s.w_router.to(torch.float64).T)
    choice = (score + s.bias.to(torch.float64)).view(-1, GROUPS, EXPERTS // GROUPS)
    kept = choice.topk(2, dim=2).values.sum(2).topk(TOP_GROUPS, dim=1).indices
    keep = torch.zeros(choice.shape[:2], dtype=torch.bool, device="cuda").scatter_(1, kept, True)
    ids = choice.masked_fill(~keep[:, :, None], -math.inf).flatten(1).topk(TOP_K, dim=1).indices
    w = score.gather(1, ids)
    return ids, w / (w.sum(1, keepdim=True) + 1e-20) * SCALE


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    x = s.x.to(torch.float64)
    if kind in ("expert", "host"):
        return _mlp(s.expert, x)
    if kind in ("route", "layer"):
        ids, w = _routes(s)
        if kind == "route":
            return ids.to(torch.int32), w
    else:
        ids, w = s.ids.long(), s.w.to(torch.float64)
    y = torch.zeros_like(x) if s.layer.shared is None else _mlp(s.layer.shared, x)
    for e in _resident(case):
        t, k = (ids == e).nonzero(as_tuple=True)
        if t.numel():
            y.index_add_(0, t, _mlp(s.layer.experts[e], x[t]) * w[t, k, None])
    return (y, ids.to(torch.int32), w) if kind == "layer" else y
