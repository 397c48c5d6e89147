"""The work this library is timed on, and what its results have to be.

Sizes are those of the benchmark and the tests: a layer of 256 experts, hidden
2048, intermediate 512, top-8 and one shared expert, 32 x 128 x 128 DeltaNet
states, 512 x 2048 expert matrices.  Every case is one pass through the public
entry points on tensors that a program keeps on the GPU (host arrays for the
host-pointer drop-in), with quantized blocks, activations and routings of the
benchmark's distributions.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "intel-optimized-moe-streaming_amd"))

from flash_moe_hip.dequant import dequant_device  # noqa: E402
from flash_moe_hip.layer_store import ExpertLayer  # noqa: E402
from flash_moe_hip.moe_gpu import MoeRunner  # noqa: E402
from flash_moe_hip.native_expert import DeltaState, NativeExpert  # noqa: E402
from flash_moe_hip.synthetic import random_expert, torch_random_stack  # noqa: E402

Q8_0, Q3_K, Q4_K, Q5_K, Q6_K = 8, 11, 12, 13, 14
BLOCK = {Q8_0: (32, 34), Q3_K: (256, 110), Q4_K: (256, 144), Q5_K: (256, 176), Q6_K: (256, 210)}
DEV = "cuda"


def _layer_case(op, **kw):
    case = dict(op=op, layers=1, tokens=1, hidden=2048, inter=512, experts=256, top_k=8, gate=Q4_K, down=Q6_K,
                shared="same")
    case.update(kw)
    return case


def listed():
    return [
        # the reference's own caller: one expert, one token, host buffers in and out, the FP16 graph
        dict(name="host expert q3k", op="host", hidden=2048, inter=512, gate=Q3_K, down=Q3_K),
        # one recurrent layer's decode step on its resident state
        dict(name="delta step", op="delta", heads=32, value_dim=128, key_dim=128),
        # a serving loop's decode step over resident layers, captured once and replayed (the layers together are
        # larger than the last-level cache)
        _layer_case("decode", name="decode 1 captured", layers=8, captured=True, fp16=0),
        # the reference model's Q3_K layers in the reference's decode numerics, called layer by layer
        _layer_case("decode", name="decode 1 mix fp16", layers=8, gate=Q3_K, down=Q3_K, shared="q6k", captured=False,
                    fp16=1),
        # the same step with its routing on the device
        _layer_case("routed", name="decode 1 routed", layers=8, gate=Q3_K, down=Q3_K, shared="q6k"),
        # sixteen sequences decoded together
        _layer_case("decode", name="decode 16 q3k", layers=4, tokens=16, gate=Q3_K, down=Q3_K, captured=False, fp16=0),
        # a layer whose sizes are no power of two
        _layer_case("decode", name="decode 1 odd sizes", layers=8, hidden=1536, inter=768, experts=64, top_k=6,
                    captured=False, fp16=0),
        # prompts: the benchmark's, a ragged one of FP32 tokens on the reference model's layers, a long one
        _layer_case("prefill", name="prefill 128", tokens=128, bf16=True, skew=0.0),
        _layer_case("prefill", name="prefill 509 mix fp32", tokens=509, gate=Q3_K, down=Q3_K, shared="q6k", bf16=False,
                    skew=0.5),
        _layer_case("prefill", name="prefill 4096", tokens=4096, bf16=True, skew=0.0),
        # routing a prompt
        dict(name="route 2048", op="route", tokens=2048, hidden=2048, experts=256, top_k=8),
        # one role's expert matrices of a layer to FP16
        dict(name="dequant layer q6k", op="dequant", type=Q6_K, values=256 * 512 * 2048, fp16=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["host", "delta", "decode", "decode", "routed", "prefill", "prefill", "prefill", "route",
                     "dequant"])
    if op == "host":
        t = rng.choice([(Q3_K, Q3_K), (Q4_K, Q6_K), (Q4_K, Q8_0), (Q5_K, Q5_K)])
        return dict(op=op, hidden=256 * rng.randint(1, 8), inter=256 * rng.randint(1, 4), gate=t[0], down=t[1])
    if op == "delta":
        return dict(op=op, heads=rng.randint(1, 64), value_dim=_log(rng, 16, 256), key_dim=_log(rng, 16, 256))
    if op == "route":
        return dict(op=op, tokens=_log(rng, 1, 2048), hidden=4 * _log(rng, 64, 512), experts=_log(rng, 16, 256),
                    top_k=rng.randint(1, 8))
    if op == "dequant":
        t = rng.choice(sorted(BLOCK))
        return dict(op=op, type=t, values=BLOCK[t][0] * _log(rng, 8, 2 ** 19), fp16=rng.random() < 0.7)
    gate = rng.choice([Q3_K, Q4_K, Q5_K, Q6_K])
    down = rng.choice([gate, gate, Q6_K, Q8_0])
    case = _layer_case(op, gate=gate, down=down, shared=rng.choice(["none", "same", "q6k"]),
                       experts=rng.choice([16, 60, 128, 256]), top_k=rng.randint(1, 8),
                       hidden=rng.choice([512, 1024, 2048, 2048]), inter=rng.choice([256, 512, 512, 1024]))
    if op == "prefill":
        case.update(tokens=_log(rng, 2, 3000), bf16=rng.random() < 0.5, skew=rng.choice([0.0, 0.5, 1.0]))
        if case["inter"] == 1024:
            case["tokens"] = max(2, case["tokens"] // 2)
    else:
        case["tokens"] = rng.choice([1, 1, rng.randint(2, 8), rng.randint(9, 32)])
        case["layers"] = rng.randint(1, 6) if case["tokens"] == 1 else 1
        if op == "decode":
            case.update(fp16=rng.choice([0, 1]), captured=rng.random() < 0.3)
            if rng.random() < 0.25:
                case.update(hidden=rng.choice([768, 1536, 2048]), inter=rng.choice([768, 1280]), experts=60)
    return case


# ------------------------------------------------------------------ inputs


def _shared_types(case):
    if case["shared"] == "none":
        return None
    if case["shared"] == "q6k":
        return {"gate": Q6_K, "up": Q6_K, "down": Q6_K}
    return {"gate": case["gate"], "up": case["gate"], "down": case["down"]}


def _inputs(case, seed):
    """The tensors of a case from its seed alone."""
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)

    def randn(*shape):
        return torch.randn(*shape, generator=g, device=DEV)

    op = case["op"]
    if op == "host":
        rng = np.random.default_rng(seed)
        kinds = {"gate": case["gate"], "up": case["gate"], "down": case["down"]}
        # scales at which the FP16 graph stays finite
        return {"kinds": kinds, "tensors": random_expert(rng, kinds, case["hidden"], case["inter"], scale=0.002),
                "x": rng.standard_normal(case["hidden"]).astype(np.float32)}
    if op == "delta":
        h, dv, dk = case["heads"], case["value_dim"], case["key_dim"]
        unit = torch.nn.functional.normalize
        return {"state": randn(h, dv, dk) * 0.1, "q": unit(randn(h, dk), dim=1), "k": unit(randn(h, dk), dim=1),
                "v": randn(h, dv), "beta": torch.sigmoid(randn(h)), "gate": -torch.nn.functional.softplus(randn(h))}
    if op == "dequant":
        bs, _ = BLOCK[case["type"]]
        return {"raw": torch_random_stack(case["type"], 1, 1, case["values"], generator=g, device=DEV)}
    T, H, E, k = case["tokens"], case["hidden"], case["experts"], case["top_k"]
    if op == "route":
        return {"x": randn(T, H), "w": randn(E, H) * 0.05}
    types = {"gate": case["gate"], "up": case["gate"], "down": case["down"]}
    scale = 0.002 if case.get("fp16") else 0.01
    layers = [ExpertLayer.synthetic(types, E, H, case["inter"], seed=seed * 64 + i, shared_types=_shared_types(case),
                                    scale=scale, device=DEV) for i in range(case["layers"])]
    got = {"layers": layers, "x": [randn(T, H) for _ in layers]}
    if op == "routed":
        got["w"] = [randn(E, H) * 0.05 for _ in layers]
        return got
    # a router's choices: top-k of its scores (some experts more popular than others), softmax over them
    bias = case.get("skew", 0.0) * randn(len(layers), 1, E)
    top = torch.topk(randn(len(layers), T, E) + bias, k, dim=2)
    got["ids"] = [i.to(torch.int32).contiguous() for i in top.indices]
    got["weights"] = [v.contiguous() for v in torch.softmax(top.values, dim=2)]
    if case.get("bf16"):
        got["x"] = [x.to(torch.bfloat16) for x in got["x"]]
    return got


def _decode(state):
    s = state
    return [s["runner"].decode(layer, x, i, w, fp16_graph=s["fp16"])
            for layer, x, i, w in zip(s["layers"], s["x"], s["ids"], s["weights"])]


def prepare(case, seed):
    state = dict(_inputs(case, seed), op=case["op"])
    op = case["op"]
    if op == "host":
        state.update(expert=NativeExpert(), hidden=case["hidden"], inter=case["inter"])
    elif op == "delta":
        state["delta"] = DeltaState(case["heads"], case["value_dim"], case["key_dim"], device=DEV, state=state["state"])
    elif op == "dequant":
        state.update(type=case["type"], dtype=torch.float16 if case["fp16"] else torch.float32)
    else:
        state.update(runner=MoeRunner(), top_k=case["top_k"], fp16=case.get("fp16", 0))
        if op == "route":
            state["layer"] = _RouterOnly(case["experts"], case["hidden"])
    if case.get("captured"):
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _decode(state)   # the runner's workspace exists before the capture
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"], stream=side):
            state["y"] = _decode(state)
    return state


class _RouterOnly:
    """What MoeRunner.route reads of a layer: its sizes."""

    def __init__(self, n_experts, hidden):
        self.n_experts, self.hidden = n_experts, hidden


def run(state):
    s, op = state, state["op"]
    if op == "host":
        return s["expert"].forward(s["tensors"], s["kinds"], s["x"], s["hidden"], s["inter"])
    if op == "delta":
        out = s["delta"].step(s["q"], s["k"], s["v"], s["beta"], s["gate"])
        return {"out": out, "state": s["delta"].state}
    if op == "dequant":
        return dequant_device(s["raw"], s["type"], dtype=s["dtype"])
    if op == "route":
        scores = torch.empty((s["x"].shape[0], s["w"].shape[0]), dtype=torch.float32, device=s["x"].device)
        ids, weights = s["runner"].route(s["layer"], s["x"], s["top_k"], router_w=s["w"], scores=scores)
        return {"ids": ids, "weights": weights, "scores": scores}
    if op == "routed":
        return [s["runner"].decode_routed(layer, x, s["top_k"], router_w=w)
                for layer, x, w in zip(s["layers"], s["x"], s["w"])]
    if op == "prefill":
        return s["runner"].prefill(s["layers"][0], s["x"][0], s["ids"][0], s["weights"][0])
    if "graph" in s:
        s["graph"].replay()
        return s["y"]
    return _decode(s)


# ------------------------------------------------------------------ work and tolerance


def _bytes(t, values):
    bs, pb = BLOCK[t]
    return values // bs * pb


def _expert_bytes(gate, down, hidden, inter):
    return 2 * _bytes(gate, hidden * inter) + _bytes(down, hidden * inter)


def work(case):
    op = case["op"]
    if op == "host":
        h, i = case["hidden"], case["inter"]
        return {"bytes": _expert_bytes(case["gate"], case["down"], h, i) + 8 * h, "flops": 6 * h * i}
    if op == "delta":
        n = case["heads"] * case["value_dim"] * case["key_dim"]
        return {"bytes": 8 * n, "flops": 7 * n}
    if op == "dequant":
        n = case["values"]
        return {"bytes": _bytes(case["type"], n) + n * (2 if case["fp16"] else 4), "flops": 2 * n}
    T, H, E, k = case["tokens"], case["hidden"], case["experts"], case["top_k"]
    route = {"bytes": 4 * (T * H + E * H + T * E) + 8 * T * k, "flops": 2 * T * H * E}
    if op == "route":
        return route
    # the distinct experts of T uniform top-k routings (fewer where some are more popular)
    used = E * (1 - (1 - k / E) ** T)
    weights = used * _expert_bytes(case["gate"], case["down"], H, case["inter"])
    if case["shared"] != "none":
        st = _shared_types(case)
        weights += _expert_bytes(st["gate"], st["down"], H, case["inter"])
    slots = k + (case["shared"] != "none")
    n = case["layers"]
    b = weights + T * H * (2 if case.get("bf16") else 4) + T * H * 4 + 8 * T * k
    f = 6 * T * slots * H * case["inter"]
    if op == "routed":
        b, f = b + route["bytes"], f + route["flops"]
    return {"bytes": n * b, "flops": n * f}


def tolerance(case):
    """About four times what the start's results are off their 64-bit values."""
    op = case["op"]
    if op == "dequant":
        return "exact"
    if op == "host" or case.get("fp16"):
        return {"rel": 3e-4, "max": 4e-3}   # FP16 roundings of intermediate values that fall the other way
    if op == "delta":
        return {"rel": 5e-7, "max": 2e-5}
    if op == "route":
        return {"rel": 1e-6, "max": 4e-5, "differ": 5e-4}   # experts whose scores tie to the last bits
    if op == "prefill":
        return {"rel": 1.5e-6}
    if all(n & (n - 1) == 0 for n in (case["hidden"], case["inter"])):
        return {"rel": 3e-4, "max": 4e-3}   # the decode kernels' 16-bit activations
    return {"rel": 1.5e-6}


# ------------------------------------------------------------------ the same in 64 bits


def _f16(b):
    """FP16 fields (two bytes in the last dimension) as float64 columns."""
    return b.contiguous().view(torch.float16).double()


def _values(raw, t):
    """The values of a flat uint8 tensor of blocks, float64."""
    bs, pb = BLOCK[t]
    b = raw.reshape(-1, pb)
    n = b.shape[0]
    if t == Q8_0:
        return (_f16(b[:, :2]) * b[:, 2:].contiguous().view(torch.int8).double()).reshape(-1)
    i = b.int()
    if t == Q3_K:
        hm, qs, sc, d = i[:, :32], i[:, 32:96], i[:, 96:108], _f16(b[:, 108:110])
        j = torch.arange(16, device=raw.device)
        s = ((sc[:, j % 8] >> (4 * (j // 8))) & 15) | (((sc[:, 8 + j % 4] >> (2 * (j // 4))) & 3) << 4)
        sh = torch.arange(4, device=raw.device).view(1, 1, 4, 1)
        half = torch.arange(2, device=raw.device).view(1, 2, 1, 1)
        q = (qs.view(n, 2, 1, 32) >> (2 * sh)) & 3
        q = q - 4 * (1 - ((hm.view(n, 1, 1, 32) >> (4 * half + sh)) & 1))
        return (d.view(n, 1, 1) * (s - 32).view(n, 16, 1) * q.reshape(n, 16, 16)).reshape(-1)
    if t in (Q4_K, Q5_K):
        d, dmin, s = _f16(b[:, :2]), _f16(b[:, 2:4]), i[:, 4:16]
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
        qs = i[:, -128:].view(n, 4, 1, 32)
        nib = torch.arange(2, device=raw.device).view(1, 1, 2, 1)
        q = (qs >> (4 * nib)) & 15
        if t == Q5_K:
            bit = 2 * torch.arange(4, device=raw.device).view(1, 4, 1, 1) + nib
            q = q | (((i[:, 16:48].view(n, 1, 1, 32) >> bit) & 1) << 4)
        q = q.reshape(n, 8, 32)
        return ((d * sc).view(n, 8, 1) * q - (dmin * mn).view(n, 8, 1)).reshape(-1)
    ql, qh = i[:, :128].view(n, 2, 2, 32), i[:, 128:192].view(n, 2, 1, 32)
    sc, d = b[:, 192:208].contiguous().view(torch.int8).double(), _f16(b[:, 208:210])
    lo, hi = ql & 15, ql >> 4
    two = torch.arange(2, device=raw.device).view(1, 1, 2, 1)
    q = torch.cat([lo | (((qh >> (2 * two)) & 3) << 4), hi | (((qh >> (4 + 2 * two)) & 3) << 4)], 2) - 32
    return ((d * sc).view(n, 16, 1) * q.reshape(n, 16, 16)).reshape(-1)


def _half(v):
    return v.to(torch.float16).double()


def _swiglu(x, gate, up, down, fp16):
    """[n, hidden] through one expert; fp16: rounded to FP16 where the FP16 graph rounds."""
    if not fp16:
        g, u = x @ gate.T, x @ up.T
        return (g * torch.sigmoid(g) * u) @ down.T
    # (weights round to FP32 before FP16, as the dequantizers leave them)
    gate, up, down = (_half(w.float()) for w in (gate, up, down))
    x = _half(x)
    g, u = _half(x @ gate.T), _half(x @ up.T)
    return _half(_half(_half(g * _half(torch.sigmoid(g))) * u) @ down.T)


def _matrices(tensors, types, hidden, inter):
    return [_values(tensors[r], types[r]).view(*(s for s in ((hidden, inter) if r == "down" else (inter, hidden))))
            for r in ("gate", "up", "down")]


def _layer(case, layer, x, ids, weights):
    x = x.double()
    y = torch.zeros_like(x)
    flat = ids.reshape(-1).long()
    k = ids.shape[1]
    for e in torch.unique(flat).tolist():
        at = (flat == e).nonzero().flatten()
        tensors = {r: layer.tensors[r].view(case["experts"], -1)[e] for r in ("gate", "up", "down")}
        m = _matrices(tensors, {"gate": case["gate"], "up": case["gate"], "down": case["down"]}, case["hidden"],
                      case["inter"])
        out = _swiglu(x[at // k], *m, case.get("fp16"))
        y.index_add_(0, at // k, out * weights.reshape(-1)[at].double().unsqueeze(1))
    if case["shared"] != "none":
        s = layer.shared
        m = _matrices({"gate": s.gate, "up": s.up, "down": s.down}, _shared_types(case), case["hidden"], case["inter"])
        y += torch.sigmoid(x @ s.gate_inp.double()).unsqueeze(1) * _swiglu(x, *m, 0)
    return y


def _route(x, w, k):
    scores = x.double() @ w.double().T
    top = torch.topk(scores, k, dim=1)
    return scores, top.indices.to(torch.int32), torch.softmax(top.values, dim=1)


def exact(case, seed):
    v, op = _inputs(case, seed), case["op"]
    if op == "host":
        m = _matrices({r: torch.from_numpy(np.asarray(t)).to(DEV) for r, t in v["tensors"].items()}, v["kinds"],
                      case["hidden"], case["inter"])
        return _swiglu(torch.from_numpy(v["x"]).to(DEV).double().view(1, -1), *m, 1).view(-1)
    if op == "delta":
        q, k, val, s = (v[n].double() for n in ("q", "k", "v", "state"))
        s = s * torch.exp(v["gate"].double()).view(-1, 1, 1)
        delta = v["beta"].double().view(-1, 1) * (val - (s * k.unsqueeze(1)).sum(2))
        s = s + delta.unsqueeze(2) * k.unsqueeze(1)
        return {"out": (s * q.unsqueeze(1)).sum(2), "state": s}
    if op == "dequant":
        return _values(v["raw"], case["type"])
    if op == "route":
        scores, _, weights = _route(v["x"], v["w"], case["top_k"])
        return {"ids": None, "weights": weights, "scores": scores}
    got = []
    for n, layer in enumerate(v["layers"]):
        x = v["x"][n]
        if op == "routed":
            _, ids, weights = _route(x, v["w"][n], case["top_k"])
            got.append((_layer(case, layer, x, ids, weights), None, weights))
        else:
            got.append(_layer(case, layer, x, v["ids"][n], v["weights"][n]))
    return got[0] if op == "prefill" else got
