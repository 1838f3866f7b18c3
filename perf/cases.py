"""The work that is timed: MoE feed-forward blocks and affine linears, from one token to 4096.

A case is one of two calls on a short stack of independently drawn layers:

* ``block``: a MoE block per layer, as ``forward`` (router, experts, combine,
  residual), ``rmsnorm`` (the same with the post-attention RMSNorm in front)
  or ``experts`` (the expert hook: routes are given);
* ``linear``: the four square attention projections of a layer
  (``native_affine_qmm``).

Geometries, storage types, code widths and routers are those of
``trifuse_amd.workload``; decode steps run sixteen layers, as its timing loop
does, so that the weights come from memory and not from a cache. Steps that a
serving program would record once and replay (``graph``) are captured into a
HIP graph beforehand, with the inputs in place; all other passes call the
library from Python each time.
"""
import math

import torch

from trifuse_amd import moe

GEOMETRY = {"olmoe": (2048, 1024, 64, 8), "granite": (1536, 512, 40, 8)}  # hidden, intermediate, experts, top k
EPS = 1e-5


def block(name, geometry, tokens, layers, call="forward", bits=4, dtype="bf16", router="dense", zipf=False,
          graph=False):
    return {"name": name, "kind": "block", "geometry": geometry, "tokens": tokens, "layers": layers, "call": call,
            "bits": bits, "dtype": dtype, "router": router, "zipf": zipf, "graph": graph}


def linear(name, width, rows, layers, bits=4, dtype="bf16", graph=False):
    return {"name": name, "kind": "linear", "width": width, "rows": rows, "layers": layers, "bits": bits,
            "dtype": dtype, "graph": graph}


def listed():
    return [
        # One sequence being decoded: a replayed step, bound by launches and latency.
        block("olmoe decode 1", "olmoe", 1, 16, graph=True),
        # A few sequences, packs as shipped (half, affine router), norm fused in, called eagerly.
        block("olmoe decode 5 half", "olmoe", 5, 16, call="rmsnorm", dtype="f16", router="affine"),
        # A small serving batch.
        block("olmoe decode 8", "olmoe", 8, 16, graph=True),
        # The same batch on 8-bit experts.
        block("olmoe decode 8 int8", "olmoe", 8, 16, bits=8, graph=True),
        # A serving batch of the smaller model.
        block("granite decode 32", "granite", 32, 16, graph=True),
        # A larger, odd batch through the expert hook, whose caller has routed the tokens.
        block("olmoe batch 45 hook", "olmoe", 45, 16, call="experts", graph=True),
        # A short prompt on 8-bit experts.
        block("olmoe prefill 300 int8", "olmoe", 300, 2, bits=8),
        # An ordinary prompt.
        block("olmoe prefill 512", "olmoe", 512, 2),
        # An odd prompt on the shipped packs with the norm fused in.
        block("olmoe prefill 1111 half", "olmoe", 1111, 2, call="rmsnorm", dtype="f16", router="affine"),
        # A long prompt of the smaller model.
        block("granite prefill 2048", "granite", 2048, 2),
        # The longest prompt, with a few experts much more popular than the others.
        block("olmoe prefill 4096 zipf", "olmoe", 4096, 2, zipf=True),
        # Attention projections of a prompt.
        linear("linear 1024", 2048, 1024, 2),
    ]


def draw(rng):
    if rng.random() < 0.12:
        width = rng.choice([1536, 2048])
        rows = round(math.exp(rng.uniform(0, math.log(2048))))
        small = rows <= 64
        return {k: v for k, v in linear("", width, rows, 8 if small else 2, bits=rng.choice([4, 4, 8]),
                                        dtype=rng.choice(["bf16", "f16"]), graph=small).items() if k != "name"}
    geometry = rng.choice(["olmoe", "olmoe", "granite"])
    bits = rng.choice([4, 4, 4, 8])
    dtype = rng.choice(["bf16", "bf16", "f16"])
    tokens = round(math.exp(rng.uniform(0, math.log(4000 if bits == 4 else 1500))))
    small = tokens <= 64
    case = block("", geometry, tokens, 16 if small else 2, call=rng.choice(["forward", "forward", "rmsnorm", "experts"]),
                 bits=bits, dtype=dtype, router="affine" if dtype == "f16" else "dense",
                 zipf=not small and rng.random() < 0.3, graph=small and rng.random() < 0.8)
    del case["name"]
    return case


# -- inputs ------------------------------------------------------------------

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _dtype(case):
    return torch.float16 if case["dtype"] == "f16" else torch.bfloat16


def _affine(gen, lead, rows, width, bits, dtype, scale=1.0):
    """Packed codes uniform over their range, group scales over a factor of four, and biases near
    the middle of the range, so that the weights are about centred on zero."""
    q = torch.randint(-2 ** 31, 2 ** 31, (*lead, rows, width * bits // 32), generator=gen, device="cuda",
                      dtype=torch.int32)
    u = torch.rand((*lead, rows, width // 64), generator=gen, device="cuda")
    s = ((0.005 + 0.015 * u) * scale * (16.0 / 2 ** bits)).to(dtype)
    off = 2 ** (bits - 1) + torch.rand(u.shape, generator=gen, device="cuda") - 1.0
    return q, s, (-s.float() * off).to(dtype)


def _normal(gen, shape, dtype, sigma=1.0):
    return (torch.randn(shape, generator=gen, device="cuda") * sigma).to(dtype)


def _inputs(case, seed):
    gen, dtype = _generator(seed), _dtype(case)
    if case["kind"] == "linear":
        n = case["width"]
        return [{"x": _normal(gen, (case["rows"], n), dtype),
                 "w": [_affine(gen, (), n, n, case["bits"], dtype) for _ in range(4)]} for _ in range(case["layers"])]
    H, I, E, K = GEOMETRY[case["geometry"]]
    T, layers = case["tokens"], []
    for _ in range(case["layers"]):
        one = {"x": _normal(gen, (T, H), dtype), "residual": _normal(gen, (T, H), dtype)}
        for proj, (rows, width) in (("gate", (I, H)), ("up", (I, H)), ("down", (H, I))):
            one[proj] = _affine(gen, (E,), rows, width, case["bits"], dtype)
        if case["router"] == "affine":
            one["router"] = _affine(gen, (), E, H, 4, dtype, scale=0.35)
        else:
            one["router"] = _normal(gen, (E, H), dtype, 0.02)
        one["bias"] = None
        if case["zipf"]:
            rank = torch.randperm(E, generator=gen, device="cuda") + 1
            one["bias"] = -0.875 * 1.1 * torch.log(rank.float())
        if case["call"] == "rmsnorm":
            one["norm"] = _normal(gen, (H,), dtype, 0.1) + 1
        if case["call"] == "experts":
            logits = torch.randn((T, E), generator=gen, device="cuda")
            one["gates"], idx = torch.softmax(logits, -1).topk(K, dim=-1)
            one["idx"] = idx.to(torch.int32)
        layers.append(one)
    return layers


class State:
    pass


def prepare(case, seed):
    state = State()
    state.case, state.layers, state.graph = case, _inputs(case, seed), None
    if case["kind"] == "block":
        H, I, E, K = GEOMETRY[case["geometry"]]
        state.block = moe.MoEBlock(H, I, E, K, route=case["geometry"], bits=case["bits"], dtype=_dtype(case),
                                   router=case["router"], residual_multiplier=1.0 if case["geometry"] == "olmoe" else 0.22)
        for one in state.layers:
            affine = case["router"] == "affine"
            rq, rs, rb = one["router"] if affine else (None, None, None)
            one["weights"] = moe.ExpertWeights(None if affine else one["router"], *one["gate"], *one["up"],
                                               *one["down"], logit_bias=one["bias"], router_q=rq, router_s=rs,
                                               router_b=rb)
    if case["graph"]:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _step(state)
        torch.cuda.current_stream().wait_stream(side)
        state.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state.graph):
            state.out = _step(state)
    return state


def _step(state):
    case, out = state.case, []
    for one in state.layers:
        if case["kind"] == "linear":
            out.append([moe.native_affine_qmm(one["x"], q, s, b, 64, case["bits"]) for q, s, b in one["w"]])
        elif case["call"] == "rmsnorm":
            out.append(state.block.forward_rmsnorm(one["x"], one["weights"], one["norm"], EPS))
        elif case["call"] == "experts":
            out.append(state.block.experts(one["x"], one["idx"], one["gates"], one["weights"], one["residual"]))
        else:
            out.append(state.block.forward(one["x"], one["weights"], one["residual"]))
    return out


def run(state):
    if state.graph is None:
        return _step(state)
    state.graph.replay()
    return state.out


# -- what a pass cannot do without -------------------------------------------

def _packed_bytes(rows, width, bits):
    return rows * width * bits // 8 + 2 * rows * (width // 64) * 2


def work(case):
    if case["kind"] == "linear":
        n, rows = case["width"], case["rows"]
        return {"bytes": case["layers"] * 4 * (_packed_bytes(n, n, case["bits"]) + 2 * rows * n * 2),
                "flops": case["layers"] * 4 * 2 * rows * n * n}
    H, I, E, K = GEOMETRY[case["geometry"]]
    T = case["tokens"]
    # Experts that T tokens reach when each picks K of E at random; popular experts change little,
    # because they come with enough tokens to reach the others.
    reached = E * (1 - (1 - K / E) ** T)
    per_expert = 2 * _packed_bytes(I, H, case["bits"]) + _packed_bytes(H, I, case["bits"])
    router = 0 if case["call"] == "experts" else _packed_bytes(E, H, 4) if case["router"] == "affine" else E * H * 2
    streams = 2 if case["call"] == "rmsnorm" else 3  # x, the residual unless it is x, and y
    return {"bytes": case["layers"] * (reached * per_expert + router + streams * T * H * 2),
            "flops": case["layers"] * (2 * T * K * 3 * H * I + (0 if case["call"] == "experts" else 2 * T * H * E))}


# -- the same in 64 bits -----------------------------------------------------

def _dequant(q, s, b, bits):
    shift = torch.arange(0, 32, bits, device=q.device, dtype=torch.int32)
    codes = (q.unsqueeze(-1) >> shift) & (2 ** bits - 1)
    codes = codes.reshape(*q.shape[:-1], -1, 64).double()
    return (codes * s.double().unsqueeze(-1) + b.double().unsqueeze(-1)).flatten(-2)


def _exact_block(case, one):
    H, I, E, K = GEOMETRY[case["geometry"]]
    dtype, x = _dtype(case), one["x"].double()
    residual = one["residual"].double()
    if case["call"] == "rmsnorm":
        # The block takes the norm's result in the storage type.
        residual = x
        x = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS)
        x = (x.to(dtype).double() * one["norm"].double()).to(dtype).double()
    if case["call"] == "experts":
        idx, gates = one["idx"].long(), one["gates"].double()
    else:
        # Routing is a choice among values in the storage type: the router, the logits and the
        # probabilities are rounded to it where the definition of the path says so.
        router = one["router"]
        router = _dequant(*router, 4).to(dtype) if case["router"] == "affine" else router
        logits = x @ router.double().T
        if one["bias"] is not None:
            logits = logits + one["bias"].double()
        logits = logits.to(dtype)
        if case["geometry"] == "olmoe":
            prob = torch.softmax(logits.double(), -1).to(dtype)
            idx = torch.sort(prob.float(), dim=-1, descending=True, stable=True).indices[:, :K]
            gates = prob.gather(1, idx).double()
        else:
            idx = torch.sort(logits.float(), dim=-1, stable=True).indices[:, -K:]
            gates = torch.softmax(logits.gather(1, idx).double(), -1)
    total = torch.zeros_like(x)
    for e in range(E):
        token, slot = (idx == e).nonzero(as_tuple=True)
        if token.numel():
            gate, up, down = (_dequant(*(t[e] for t in one[p]), case["bits"]) for p in ("gate", "up", "down"))
            rows = x[token]
            hidden = torch.nn.functional.silu(rows @ gate.T) * (rows @ up.T)
            total.index_add_(0, token, (hidden @ down.T) * gates[token, slot].unsqueeze(-1))
    return residual + (1.0 if case["geometry"] == "olmoe" else 0.22) * total


def exact(case, seed):
    out = []
    for one in _inputs(case, seed):
        if case["kind"] == "linear":
            out.append([one["x"].double() @ _dequant(q, s, b, case["bits"]).T for q, s, b in one["w"]])
        else:
            out.append(_exact_block(case, one))
    return out


def tolerance(case):
    # Measured against exact(): bf16 0.0021 to 0.0037 (weights or hidden rows rounded to 8 bits, sums
    # in 32), half 0.00027 to 0.00044.
    return {"rel": 2e-3 if case["dtype"] == "f16" else 1e-2}
