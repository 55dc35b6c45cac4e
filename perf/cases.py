"""Timed cases of the quantized mixture-of-experts path, through its public
entry points: what a serving program runs per decode step and per prefill
chunk.

Kinds of case (``case["kind"]``):

``block``   :class:`titan_amd.moe_block.SparseMoeBlock`, the routed block as one
            call.  Up to 16 tokens it is the MoE part of a decode step over
            several layers, captured once in a HIP graph and replayed, as a
            serving loop does (each layer has its own weights and its own
            hidden states, since the attention between two layers is not part
            of this path).  Above, one eager call of one layer: a prefill chunk.
``dense``   :func:`titan_amd.ops.quantized_matmul` over the dense projections
            of several layers, for a batch of decoding sequences (captured).
``fused``   :func:`titan_amd.ops.gate_up_silu` and :func:`titan_amd.ops.down_wsum`
            over MLX-layout weights: the decode step of a program that keeps
            the checkpoint's own layout (captured).
``glu``     :class:`titan_amd.switch_layers.SwitchGLU`, the drop-in layer, with
            the overlays installed and the weights warmed up (eager).
``int8``    the opt-in int8-activation x int4-weight gather over expert-sorted
            rows (eager).

Weights are random 4-bit (or 8-bit) affine codes whose bias centres them, as
the quantisation of a zero-mean weight gives, scaled for activations of unit
variance; a router column gives some experts more tokens than others.
"""

import math

import torch

from titan_amd import ops, patches
from titan_amd.kernels import moe_gather_int8
from titan_amd.moe_block import SharedExpert, SparseMoeBlock
from titan_amd.patches import gather_ws
from titan_amd.switch_layers import QuantizedSwitchLinear, SwitchGLU

DEV = "cuda"
GROUP = 64

# routed-expert shapes: experts, experts per token, hidden, intermediate
FINE = {"E": 256, "k": 10, "H": 2048, "I": 512}
WIDE = {"E": 128, "k": 8, "H": 2048, "I": 768}
# dense projections: output rows, input columns
DENSE = ((4096, 2048), (2048, 4096), (9216, 2048), (1000, 2048), (5120, 2560))


def _block(T, layers, shared, router, shape=FINE):
    return {"kind": "block", "T": T, "layers": layers, "shared": shared, "router": router, **shape}


def listed():
    cases = {
        # one decoding sequence through the dense projections of eight layers
        "dense_4bit_1": {"kind": "dense", "M": 1, "N": 4096, "K": 2048, "bits": 4, "group": 64, "layers": 8},
        # a decode batch of 24 sequences through 8-bit projections (the layers kept at 8 bits)
        "dense_8bit_24": {"kind": "dense", "M": 24, "N": 4096, "K": 2048, "bits": 8, "group": 64, "layers": 8},
        # single-user decoding: latency of the MoE part of six layers, one token each
        "block_1": _block(1, 6, True, "q8"),
        # speculative verification or a small batch, still on the decode kernels (40 pairs)
        "block_4": _block(4, 6, True, "q8"),
        # the other routed shape, no shared expert, unquantised router, decoding from MLX-layout weights
        "block_3_wide": _block(3, 6, False, "bf16", WIDE),
        # a decode batch of 16: 160 pairs, past the sort threshold
        "block_16": _block(16, 4, True, "q8"),
        # a short prompt, or a chunk of one: fewer than four rows per expert
        "block_96": _block(96, 1, True, "q8"),
        # a ragged prompt of ordinary length
        "block_777": _block(777, 1, False, "bf16"),
        # a full prefill chunk
        "block_4096": _block(4096, 1, True, "bf16"),
        # eight decoding sequences on MLX-layout weights
        "fused_8": {"kind": "fused", "T": 8, "layers": 6, **FINE},
        # a prefill chunk through the drop-in layer
        "glu_512": {"kind": "glu", "T": 512, **FINE},
        # a prefill chunk's gate_up through the int8 path
        "int8_2048": {"kind": "int8", "T": 2048, **FINE},
    }
    return [{"name": n, **c} for n, c in cases.items()]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)) - 0.2)))))


def draw(rng):
    kind = rng.choice(("block", "block", "block", "block", "dense", "dense", "fused", "glu", "int8"))
    if kind == "dense":
        N, K = rng.choice(DENSE)
        return {"kind": "dense", "M": _log_int(rng, 1, 64), "N": N, "K": K, "bits": rng.choice((4, 8)),
                "group": rng.choice((32, 64, 64, 128)), "layers": 8}
    shape = rng.choice((FINE, FINE, WIDE))
    if kind == "block":
        shared, router = rng.random() < 0.5, rng.choice(("bf16", "q8", "q4"))
        if rng.random() < 0.5:
            return _block(rng.randint(1, 16), 4, shared, router, shape)
        return _block(_log_int(rng, 17, 4000), 1, shared, router, shape)
    if kind == "fused":
        return {"kind": "fused", "T": rng.randint(1, 16), "layers": 4, **shape}
    if kind == "glu":
        return {"kind": "glu", "T": _log_int(rng, 2, 1024), **shape}
    return {"kind": "int8", "T": _log_int(rng, 64, 2048), **FINE}


# ------------------------------------------------------------------ inputs


def _gen(seed, salt=0):
    return torch.Generator(device=DEV).manual_seed(seed * 1000003 + salt)


def _quant(g, lead, K, bits=4, group=GROUP, gain=1.0):
    """(words, scales, biases) of a quantised zero-mean weight [*lead, K] whose
    rows have norm ``gain``: the codes' bias is about minus half their range."""
    levels = 2 ** bits
    step = gain * math.sqrt(12.0 / K) / levels
    w = torch.randint(-2 ** 31, 2 ** 31, (*lead, K * bits // 32), dtype=torch.int32, device=DEV, generator=g)
    u = torch.rand(*lead, K // group, device=DEV, generator=g)
    s = (step * (0.7 + 0.6 * u)).to(torch.bfloat16)
    v = torch.rand(*lead, K // group, device=DEV, generator=g)
    b = (-s.float() * (levels - 1) * (0.48 + 0.04 * v)).to(torch.bfloat16)
    return w, s, b


def _tokens(g, T, H):
    x = torch.randn(T, H, device=DEV, generator=g)
    x[:, 0] = 1.0  # the direction that the router's popularity column reads
    return x.to(torch.bfloat16)


def _router(g, case):
    E, H = case["E"], case["H"]
    if case["router"] != "bf16":
        w, s, b = _quant(g, (E,), H, int(case["router"][1:]), gain=1.5)
        return w, s, b
    w = torch.randn(E, H, device=DEV, generator=g) / math.sqrt(H)
    w[:, 0] = 0.6 * torch.randn(E, device=DEV, generator=g)
    return w.to(torch.bfloat16)


def _layer(case, seed, layer):
    """One layer's tensors: hidden states, router, routed and shared experts."""
    g = _gen(seed, layer)
    E, H, I = case["E"], case["H"], case["I"]
    d = {"x": _tokens(g, case["T"], H), "gate_up": _quant(g, (E, 2 * I), H, gain=1.2),
         "down": _quant(g, (E, H), I, gain=1.0)}
    if "router" in case:
        d["router"] = _router(g, case)
    if case.get("shared"):
        d["sh_gate_up"] = _quant(g, (1, 2 * I), H, gain=1.2)
        d["sh_down"] = _quant(g, (1, H), I, gain=1.0)
        d["sh_gate"] = (torch.randn(1, H, device=DEV, generator=g) / math.sqrt(H)).to(torch.bfloat16)
    return d


def _routing(g, case, T):
    """Distinct experts per token with uneven popularity, and softmax scores."""
    logits = torch.randn(T, case["E"], device=DEV, generator=g) + 0.6 * torch.randn(case["E"], device=DEV, generator=g)
    top, idx = logits.topk(case["k"], dim=-1)
    return idx.to(torch.int32), torch.softmax(top, dim=-1)


def _glu_inputs(case, seed):
    d = _layer(case, seed, 0)
    d["idx"], _ = _routing(_gen(seed, 77), case, case["T"])
    return d


def _int8_inputs(case, seed):
    g = _gen(seed)
    T, k, H = case["T"], case["k"], case["H"]
    x = torch.randn(T, H, device=DEV, generator=g)
    x = torch.where(torch.rand(T, H, device=DEV, generator=g) < 1e-3, x * 20.0, x).to(torch.bfloat16)
    idx, _ = _routing(g, case, T)
    ids, order = torch.sort(idx.reshape(-1), stable=True)
    return x[order // k].contiguous(), ids.contiguous(), _quant(g, (case["E"], 2 * case["I"]), H, gain=1.2)


def _dense_inputs(case, seed, layer):
    g = _gen(seed, layer)
    x = torch.randn(case["M"], case["K"], device=DEV, generator=g).to(torch.bfloat16)
    return x, _quant(g, (case["N"],), case["K"], case["bits"], case["group"])


def _captured(step):
    """``step`` once outside a capture, then captured: (graph, its outputs)."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    return {"graph": graph, "out": out, "step": step}


# --------------------------------------------------------- prepare and run


def prepare(case, seed):
    kind = case["kind"]
    if kind == "block":
        calls = []
        for layer in range(case["layers"]):
            d = _layer(case, seed, layer)
            sh = SharedExpert(d["sh_gate_up"], d["sh_down"], d["sh_gate"]) if case["shared"] else None
            quant = (GROUP, int(case["router"][1:])) if case["router"] != "bf16" else (GROUP, 4)
            calls.append((SparseMoeBlock(d["router"], d["gate_up"], d["down"], case["k"], shared=sh,
                                         router_quant=quant), d["x"]))
        if case["T"] > 16:
            return {"calls": calls}
        return _captured(lambda: [block(x) for block, x in calls])
    if kind == "dense":
        ins = [_dense_inputs(case, seed, layer) for layer in range(case["layers"])]
        return _captured(lambda: [ops.quantized_matmul(x, *w, group_size=case["group"], bits=case["bits"])
                                  for x, w in ins])
    if kind == "fused":
        ins = []
        for layer in range(case["layers"]):
            d = _layer(case, seed, layer)
            ins.append((d["x"], d["gate_up"], d["down"], *_routing(_gen(seed, 100 + layer), case, case["T"])))

        def step():
            return [ops.down_wsum(ops.gate_up_silu(x, *gu, idx), *dn, idx, sc) for x, gu, dn, idx, sc in ins]

        return _captured(step)
    if kind == "glu":
        d = _glu_inputs(case, seed)
        patches.install()
        layer = SwitchGLU(QuantizedSwitchLinear(*d["down"]), QuantizedSwitchLinear(*d["gate_up"]))
        gather_ws.warmup(layer)
        return {"glu": layer, "x": d["x"], "idx": d["idx"]}
    x, ids, w = _int8_inputs(case, seed)
    return {"int8": (x.unsqueeze(1), *w, ids, moe_gather_int8.build_tables(*w))}


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    if "calls" in state:
        return [block(x) for block, x in state["calls"]]
    if "glu" in state:
        return state["glu"](state["x"], state["idx"])
    return moe_gather_int8.OP.fast(*state["int8"])


# ------------------------------------------------------- work and tolerance


def _qbytes(rows, K, bits=4, group=GROUP):
    return rows * (K * bits / 8 + 4 * K / group)


def work(case):
    if case["kind"] == "dense":
        M, N, K = case["M"], case["N"], case["K"]
        one = _qbytes(N, K, case["bits"], case["group"]) + 2 * M * (N + K)
        return {"bytes": case["layers"] * one, "flops": case["layers"] * 2.0 * M * N * K}
    T, E, k, H, I = (case[f] for f in ("T", "E", "k", "H", "I"))
    used = E * (1.0 - (1.0 - k / E) ** T)  # experts that T tokens reach
    gate_up, down = _qbytes(2 * I, H), _qbytes(H, I)
    if case["kind"] == "int8":
        return {"bytes": used * gate_up + T * k * (2 * H + 4 + 2 * 2 * I), "flops": 2.0 * T * k * H * 2 * I}
    flops = 2.0 * T * k * 3 * H * I
    if case["kind"] == "glu":
        return {"bytes": used * (gate_up + down) + 2 * T * H + 4 * T * k + 2 * T * k * H, "flops": flops}
    bytes_ = used * (gate_up + down) + 2 * 2 * T * H
    if case["kind"] == "block":
        flops += 2.0 * T * E * H
        bytes_ += 2 * E * H if case["router"] == "bf16" or T > 16 else _qbytes(E, H, int(case["router"][1:]))
        if case["shared"]:
            flops += 2.0 * T * (3 * H * I + H)
            bytes_ += gate_up + down + 2 * H
    else:
        bytes_ += 8 * T * k
    return {"bytes": case["layers"] * bytes_, "flops": case["layers"] * flops}


def tolerance(case):
    # bf16 outputs (half an ULP is 2e-3 of a value) of sums in 32 bits.
    # dense and int8 round once; the other kinds also round the intermediate
    # h, and past the sort threshold each expert's output, to bf16.
    if case["kind"] in ("dense", "int8"):
        return {"rel": 6e-3}
    return {"rel": 1e-2}


# ----------------------------------------------------------- 64-bit results


def _dequant(q, bits=4, group=GROUP, rounded=False):
    """The weight in 64 bits; ``rounded``: through bf16, as the sorted path defines it."""
    w, s, b = q
    shifts = torch.arange(0, 32, bits, device=w.device, dtype=torch.int32)
    codes = (w.unsqueeze(-1) >> shifts) & (2 ** bits - 1)
    codes = codes.reshape(*w.shape[:-1], -1).double()
    out = codes * s.double().repeat_interleave(group, -1) + b.double().repeat_interleave(group, -1)
    return out.float().to(torch.bfloat16).double() if rounded else out


def _expert(q, e):
    return tuple(t[e] for t in q)


def _mlp(x, gate_up, down, rounded):
    gu = x @ _dequant(gate_up, rounded=rounded).t()
    gate, up = gu.chunk(2, dim=-1)
    return (torch.nn.functional.silu(gate) * up) @ _dequant(down, rounded=rounded).t()


def _experts(x, idx, gate_up, down, rounded):
    """Every (token, slot) pair's expert output [T, k, H]."""
    T, k = idx.shape
    flat = idx.reshape(-1).long()
    out = torch.empty(T * k, x.shape[1], dtype=torch.float64, device=x.device)
    for e in flat.unique().tolist():
        rows = (flat == e).nonzero().reshape(-1)
        out[rows] = _mlp(x[rows // k], _expert(gate_up, e), _expert(down, e), rounded)
    return out.reshape(T, k, -1)


def _exact_block(case, seed, layer):
    d = _layer(case, seed, layer)
    x, T = d["x"].double(), case["T"]
    batch = T > 16  # beyond, dense layers read weights rounded to bf16
    if case["router"] == "bf16":
        router = d["router"].double()
    else:
        router = _dequant(d["router"], int(case["router"][1:]), rounded=batch)
    top, idx = (x @ router.t()).topk(case["k"], dim=-1)
    scores = torch.softmax(top, dim=-1)
    y = _experts(x, idx, d["gate_up"], d["down"], T * case["k"] >= 64)
    y = (y * scores.unsqueeze(-1)).sum(1)
    if case["shared"]:
        sh = _mlp(x, _expert(d["sh_gate_up"], 0), _expert(d["sh_down"], 0), batch)
        y = y + torch.sigmoid(x @ d["sh_gate"].double().t()) * sh
    return y


def exact(case, seed):
    kind = case["kind"]
    if kind == "block":
        return [_exact_block(case, seed, layer) for layer in range(case["layers"])]
    if kind == "dense":
        out = []
        for layer in range(case["layers"]):
            x, w = _dense_inputs(case, seed, layer)
            out.append(x.double() @ _dequant(w, case["bits"], case["group"]).t())
        return out
    if kind == "fused":
        out = []
        for layer in range(case["layers"]):
            d = _layer(case, seed, layer)
            idx, scores = _routing(_gen(seed, 100 + layer), case, case["T"])
            y = _experts(d["x"].double(), idx, d["gate_up"], d["down"], False)
            out.append((y * scores.double().unsqueeze(-1)).sum(1))
        return out
    if kind == "glu":
        d = _glu_inputs(case, seed)
        return _experts(d["x"].double(), d["idx"], d["gate_up"], d["down"], case["T"] * case["k"] >= 64)
    x, ids, w = _int8_inputs(case, seed)
    # per-token symmetric int8: the scale in fp32, the codes to nearest even
    sx = x.float().abs().amax(-1, keepdim=True) / 127.0
    xi = torch.clamp(torch.round(x.float() / sx), -127, 127).double() * sx.double()
    out = torch.empty(x.shape[0], w[0].shape[1], dtype=torch.float64, device=x.device)
    for e in ids.unique().tolist():
        rows = (ids == e).nonzero().reshape(-1)
        out[rows] = xi[rows] @ _dequant(_expert(w, e)).t()
    return out.unsqueeze(1)
