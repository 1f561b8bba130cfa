"""The work that is timed: the MoE layer of Qwen3.6-35B-A3B from one decoded token to a prefill chunk, the quantized
projections around it (GGMLWeight through F.linear, linear_mfma) and dequantization, through the package's own entry
points on seeded synthetic weights.

Kinds of case:
  step     one decode step's MoE halves, x <- x + MoE(rms_norm(x)), layer after layer on one workspace, captured as
           one graph and replayed (the model's loop at 1 .. 8 tokens; every call runs on one stream)
  batch    one batched decode step's MoE layers on the same tokens, launched eagerly inside one fork scope
  prefill  one MoE layer on a prompt (or a chunk of one), launched eagerly
  project  one decode step's projections: F.linear(x, GGMLWeight) of `count` weights, one graph, at most 8 tokens
  linear   linear_mfma: a projection above 8 tokens without a dequantized copy of the weight
  dequant  dequantize_gpu: a weight's bf16 (or fp32) values, as a program that keeps dense weights makes them

Weights follow gguf.synth's block recipes and are made on the GPU from the seed."""
import contextlib
import math
import os
import random
import sys

import numpy as np
import torch
import torch.nn.functional as F

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "willow-v2_amd"))

from gguf import hip  # noqa: E402
from gguf.hip.moe import MoELayer, new_workspace  # noqa: E402

BLOCK_BYTES = {"Q4_K": 144, "Q6_K": 210}
HIDDEN, INTER = 2048, 512


def _moe(kind, tokens, layers, down="Q6_K", gate_up="Q4_K", experts=256, top_k=8, zipf=False, bf16=False):
    return {"kind": kind, "tokens": tokens, "layers": layers, "gate_up": gate_up, "down": down, "experts": experts,
            "top_k": top_k, "zipf": zipf, "bf16": bf16}


def _matrix(kind, weight, rows, k, tokens=0, count=1, bf16=True):
    return {"kind": kind, "type": weight, "rows": rows, "k": k, "tokens": tokens, "count": count, "bf16": bf16}


def listed():
    return [
        # interactive decoding: one token through eight layers of the model's loop
        dict(_moe("step", 1, 8), name="step_1"),
        # a handful of concurrent users, an odd count; every expert holds a token or two
        dict(_moe("step", 5, 4), name="step_5"),
        # batched serving, uniform routing: ~100 experts of one or two tokens each
        dict(_moe("batch", 16, 4), name="batch_16"),
        # batched serving with skewed expert popularity, the benchmark's batched-decode workload
        dict(_moe("batch", 64, 4, zipf=True), name="batch_64_zipf"),
        # a short ragged prompt in the model's own bf16: about nine tokens per expert; a layer with Q4_K down weights
        # (Q4_K_M files mix the two)
        dict(_moe("prefill", 300, 1, down="Q4_K", bf16=True), name="prefill_300"),
        # a medium prompt, not a multiple of any tile
        dict(_moe("prefill", 1000, 1), name="prefill_1000"),
        # the benchmark's prefill chunk
        dict(_moe("prefill", 4096, 1), name="prefill_4096"),
        # the quantized projections of one decode step: one token in the model's bf16; eight tokens in fp32
        dict(_matrix("project", "Q4_K", 4096, 2048, 1, 24), name="project_1"),
        dict(_matrix("project", "Q6_K", 2048, 4096, 8, 12, bf16=False), name="project_8"),
        # projections of a short prompt and of a prefill chunk from the quantized blocks
        dict(_matrix("linear", "Q4_K", 4096, 2048, 200), name="linear_200"),
        dict(_matrix("linear", "Q6_K", 2048, 2048, 4096), name="linear_4096"),
        # a large projection made dense once
        dict(_matrix("dequant", "Q4_K", 8192, 2048), name="dequant_q4k"),
    ]


def _spread(rng, lo, hi):
    """A whole number from lo to hi, evenly over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng: random.Random):
    kind = rng.choice(("step", "batch", "prefill", "prefill", "project", "linear", "dequant"))
    if kind in ("step", "batch", "prefill"):
        tokens = {"step": rng.randint(1, 8), "batch": _spread(rng, 9, 64), "prefill": _spread(rng, 65, 4096)}[kind]
        layers = {"step": rng.randint(2, 6), "batch": rng.randint(1, 4), "prefill": 1}[kind]
        return _moe(kind, tokens, layers, down=rng.choice(("Q6_K", "Q6_K", "Q4_K")),
                    gate_up=rng.choice(("Q4_K", "Q4_K", "Q6_K")), experts=rng.choice((256, 256, 128, 40)),
                    top_k=rng.choice((8, 8, 6, 4)), zipf=rng.random() < 0.4, bf16=rng.random() < 0.3)
    weight = rng.choice(("Q4_K", "Q6_K"))
    k = 256 * _spread(rng, 2, 16)
    if kind == "project":  # any number of rows
        return _matrix(kind, weight, _spread(rng, 200, 8192), k, rng.randint(1, 8), rng.randint(4, 16),
                       rng.random() < 0.5)
    if kind == "linear":
        return _matrix(kind, weight, 256 * _spread(rng, 2, 16), k, _spread(rng, 9, 4096))
    return _matrix(kind, weight, _spread(rng, 200, 8192), k, bf16=rng.random() < 0.7)


# --- inputs ----------------------------------------------------------------------------------------------------------

def _blocks(weight, n, gen):
    """n random blocks (gguf.synth's recipes): uint8 [n, block bytes]."""
    b = torch.randint(0, 256, (n, BLOCK_BYTES[weight]), dtype=torch.uint8, device="cuda", generator=gen)
    f16_at = (0, 2) if weight == "Q4_K" else (208,)
    if weight == "Q6_K":
        b[:, 192:208] = torch.randint(-32, 32, (n, 16), dtype=torch.int8, device="cuda", generator=gen).view(torch.uint8)
    for at in f16_at:
        d = (torch.randn(n, device="cuda", generator=gen).abs() * 0.01).half()
        b[:, at:at + 2] = d.view(torch.uint8).view(n, 2)
    return b


def _generator(seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    return gen


def _raw_moe(case, gen):
    """One layer's tensors, before any layout of the package."""
    E, I = case["experts"], INTER
    raw = {
        "gate_up": _blocks(case["gate_up"], E * 2 * I * (HIDDEN // 256), gen).view(E, -1),
        "down": _blocks(case["down"], E * HIDDEN * (I // 256), gen).view(E, -1),
        "router": torch.randn(E, HIDDEN, device="cuda", generator=gen) * 0.02,
        "shared_gate_up": _blocks(case["gate_up"], 2 * I * (HIDDEN // 256), gen).view(-1),
        "shared_down": _blocks(case["down"], HIDDEN * (I // 256), gen).view(-1),
        "shared_gate": torch.randn(HIDDEN, device="cuda", generator=gen) * 0.02,
        "norm": torch.randn(HIDDEN, device="cuda", generator=gen) * 0.1,
        "bias": None,
    }
    if case["zipf"]:  # expert popularity falling as rank^-1.1
        raw["bias"] = torch.empty(E, device="cuda")
        perm = torch.randperm(E, device="cuda", generator=gen)
        raw["bias"][perm] = -1.1 * torch.log(torch.arange(1, E + 1, device="cuda", dtype=torch.float32))
    return raw


def _layer(case, raw):
    return MoELayer(gate_up=raw["gate_up"], down=raw["down"], router=raw["router"], router_bias=raw["bias"],
                    hidden=HIDDEN, inter=INTER, n_experts=case["experts"], top_k=case["top_k"],
                    gate_up_type=case["gate_up"], down_type=case["down"], shared_gate_up=raw["shared_gate_up"],
                    shared_down=raw["shared_down"], shared_gate=raw["shared_gate"], shared_inter=INTER)


def _inputs(case, seed):
    """(the raw weights, x), from the seed alone."""
    gen = _generator(seed)
    if case["kind"] in ("step", "batch", "prefill"):
        x = torch.randn(case["tokens"], HIDDEN, device="cuda", generator=gen)
        if case["bf16"]:
            x = x.bfloat16()
        return [_raw_moe(case, gen) for _ in range(case["layers"])], x
    x = torch.randn(max(case["tokens"], 1), case["k"], device="cuda", generator=gen)
    if case["bf16"]:
        x = x.bfloat16()
    n = case["rows"] * (case["k"] // 256)
    return [_blocks(case["type"], n, gen).view(-1) for _ in range(case["count"])], x


def _captured(fn):
    """fn warmed up, then captured as one graph."""
    fn()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outputs = fn()
    torch.cuda.synchronize()
    return graph, outputs


def prepare(case, seed):
    raws, x = _inputs(case, seed)
    kind = case["kind"]
    if kind in ("step", "batch", "prefill"):
        T, L = case["tokens"], case["layers"]
        layers = [_layer(case, raw) for raw in raws]
        ids = torch.empty(L, T, case["top_k"], dtype=torch.int32, device="cuda")
        wts = torch.empty(L, T, case["top_k"], device="cuda")
        if kind == "prefill":
            layers[0].workspace(T)
            return {"kind": kind, "layer": layers[0], "x": x, "ids": ids[0], "wts": wts[0]}
        ys = torch.empty(L, T, HIDDEN, device="cuda")
        if kind == "batch":
            ws = new_workspace(max(layer.workspace_bytes(T) for layer in layers), "cuda")
            return {"kind": kind, "layers": layers, "ws": ws, "x": x, "ys": ys, "ids": ids, "wts": wts}
        chain = [layer.with_norm(raw["norm"]) for layer, raw in zip(layers, raws)]
        for layer, following in zip(chain, chain[1:]):
            layer.set_next(following)
        ws = new_workspace(max(layer.workspace_bytes(T) for layer in chain), "cuda")

        def step():
            y = x
            for l, layer in enumerate(chain):
                y = layer(y, out=ys[l], ids=ids[l], weights=wts[l], workspace=ws)
            return ys, ids, wts

        graph, outputs = _captured(step)
        return {"kind": kind, "graph": graph, "outputs": outputs, "keep": (chain, layers, ws, x)}
    if kind == "project":
        weights = [hip.GGMLWeight(raw, case["type"], (case["rows"], case["k"])) for raw in raws]
        graph, outputs = _captured(lambda: [F.linear(x, w) for w in weights])
        return {"kind": kind, "graph": graph, "outputs": outputs, "keep": (weights, x)}
    return {"kind": kind, "raw": raws[0], "type": case["type"], "shape": (case["rows"], case["k"]), "x": x,
            "dtype": torch.bfloat16 if case["bf16"] else torch.float32}


def run(state):
    kind = state["kind"]
    if kind in ("step", "project"):
        state["graph"].replay()
        return state["outputs"]
    if kind == "batch":
        with hip.fork_scope("cuda") if state["layers"][0].plan(state["x"].shape[0]) == "split" else contextlib.nullcontext():
            for l, layer in enumerate(state["layers"]):
                layer(state["x"], out=state["ys"][l], ids=state["ids"][l], weights=state["wts"][l], workspace=state["ws"])
        return state["ys"], state["ids"], state["wts"]
    if kind == "prefill":
        y = state["layer"](state["x"], ids=state["ids"], weights=state["wts"])
        return y, state["ids"], state["wts"]
    if kind == "linear":
        return hip.linear_mfma(state["raw"], state["type"], state["shape"], state["x"])
    return hip.dequantize_gpu(state["raw"], state["type"], state["shape"], state["dtype"])


# --- what a pass cannot do without -----------------------------------------------------------------------------------

def _touched(case):
    """The experts that some token picks, per layer: the router's logits are N(0, 0.9) plus the bias."""
    rng = np.random.default_rng(0)
    logits = rng.standard_normal((case["tokens"], case["experts"])) * (0.02 * math.sqrt(HIDDEN))
    if case["zipf"]:
        logits -= 1.1 * np.log(np.arange(1, case["experts"] + 1))
    return len(np.unique(np.argpartition(-logits, case["top_k"] - 1, axis=1)[:, :case["top_k"]]))


def work(case):
    if case["kind"] in ("step", "batch", "prefill"):
        T, L, k = case["tokens"], case["layers"], case["top_k"]
        expert = INTER * HIDDEN // 256 * (2 * BLOCK_BYTES[case["gate_up"]] + BLOCK_BYTES[case["down"]])
        weights = (_touched(case) + 1) * expert + (case["experts"] + 1) * HIDDEN * 4
        acts = T * HIDDEN * (4 + (2 if case["bf16"] else 4)) + T * k * 8
        return {"bytes": L * (weights + acts),
                "flops": L * 2.0 * T * HIDDEN * ((k + 1) * 3 * INTER + case["experts"] + 1)}
    raw = case["rows"] * (case["k"] // 256) * BLOCK_BYTES[case["type"]]
    size = 2 if case["bf16"] else 4
    if case["kind"] == "dequant":
        return {"bytes": raw + case["rows"] * case["k"] * size, "flops": 0}
    T, n = case["tokens"], case["count"]
    return {"bytes": n * (raw + T * case["rows"] * size) + T * case["k"] * size, "flops": 2.0 * n * T * case["rows"] * case["k"]}


def tolerance(case):
    """About four times what the path differs from the same arithmetic with its sums in another order: linear_mfma and
    the GEMV against a library product on the dequantized values, the layer's GEMMs against the same experts in larger
    tiles (rel 4e-5, 6e-7, 1.2e-4; the largest differences are single bf16 roundings that fall the other way)."""
    kind = case["kind"]
    if kind == "dequant":  # each value is one rounding of an exact product and sum
        return "exact"
    if kind == "linear":  # bf16 operands and outputs
        return {"rel": 2e-4, "max": 3e-2}
    if kind == "project":  # fp32 sums; bf16 outputs may round the other way
        return {"rel": 4e-4, "max": 2.5e-2} if case["bf16"] else {"rel": 2.5e-6, "max": 2e-5}
    if kind == "step":  # fp32 throughout, layer after layer; the routing's whole values can only change at a tie
        return {"rel": 5e-6, "max": 1e-4, "differ": 1e-4}
    # experts of more than 8 tokens and the shared expert run in bf16
    return {"rel": 5e-4, "max": 3e-2, "differ": 1e-4}


# --- the same in 64 bits ---------------------------------------------------------------------------------------------

def _f16(b):
    return b.contiguous().view(torch.float16).double()


def _values(raw, weight, rows, k):
    """A matrix's dequantized values in 64 bits: [rows, k]."""
    b = raw.reshape(rows * (k // 256), BLOCK_BYTES[weight])
    n = b.shape[0]
    if weight == "Q4_K":
        d, dmin, s = _f16(b[:, 0:2]), _f16(b[:, 2:4]), b[:, 4:16].int()
        lo, mid, hi = s[:, 0:4], s[:, 4:8], s[:, 8:12]
        sc = torch.cat((lo & 63, (hi & 15) | (lo >> 6 << 4)), 1)
        m = torch.cat((mid & 63, (hi >> 4) | (mid >> 6 << 4)), 1)
        q = b[:, 16:144].reshape(n, 4, 1, 32).int()
        q = torch.cat((q & 15, q >> 4), 2).reshape(n, 8, 32).double()
        v = (d * sc).unsqueeze(2) * q - (dmin * m).unsqueeze(2)
    else:
        ql, qh = b[:, 0:128].reshape(n, 2, 2, 32).int(), b[:, 128:192].reshape(n, 2, 1, 32).int()
        low = torch.cat((ql & 15, ql >> 4), 2)  # [n, half, 4, 32]
        shift = torch.tensor([0, 2, 4, 6], device=b.device).view(1, 1, 4, 1)
        q = (low | (qh >> shift & 3) << 4).double() - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).double() * _f16(b[:, 208:210])
        v = sc.unsqueeze(2) * q.reshape(n, 16, 16)
    return v.reshape(rows, k)


def _expert(raw_gate_up, raw_down, case, x):
    gu = x @ _values(raw_gate_up, case["gate_up"], 2 * INTER, HIDDEN).T
    g, u = gu[:, :INTER], gu[:, INTER:]
    return (g * torch.sigmoid(g) * u) @ _values(raw_down, case["down"], HIDDEN, INTER).T


def _moe64(case, raw, x):
    """-> (y, weights) of one layer on x, in 64 bits."""
    logits = x @ raw["router"].double().T
    if raw["bias"] is not None:
        logits = logits + raw["bias"].double()
    p, ids = torch.topk(torch.softmax(logits, 1), case["top_k"], dim=1)
    p = p / p.sum(1, keepdim=True)
    y = torch.sigmoid(x @ raw["shared_gate"].double()).unsqueeze(1) * _expert(raw["shared_gate_up"], raw["shared_down"], case, x)
    for e in torch.unique(ids).tolist():
        t, slot = torch.nonzero(ids == e, as_tuple=True)
        y[t] += p[t, slot].unsqueeze(1) * _expert(raw["gate_up"][e], raw["down"][e], case, x[t])
    return y, p


def exact(case, seed):
    raws, x = _inputs(case, seed)
    kind = case["kind"]
    x = x.double()
    if kind in ("step", "batch", "prefill"):
        ys, ws = [], []
        for raw in raws:
            if kind == "step":
                xn = x * torch.rsqrt(x.square().mean(1, keepdim=True) + 1e-6) * (1 + raw["norm"].double())
                y, p = _moe64(case, raw, xn)
                x = x + y
                ys.append(x)
            else:
                y, p = _moe64(case, raw, x)
                ys.append(y)
            ws.append(p)
        if kind == "prefill":
            return ys[0], None, ws[0]
        return torch.stack(ys), None, torch.stack(ws)
    if kind == "project":
        return [x @ _values(raw, case["type"], case["rows"], case["k"]).T for raw in raws]
    values = _values(raws[0], case["type"], case["rows"], case["k"])
    return values if kind == "dequant" else x @ values.T
