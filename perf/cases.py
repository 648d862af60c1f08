"""The calls a user of this package has it do, as cases that can be timed and compared.

A case is a dict of plain values; ``kind`` names the public entry point it goes through:

* ``layer``   ``modeling.moe_layer.MoELayer``: gate, shared expert, routed experts, combine.
  ``mode`` "bf16" is bf16 parameters and activations; "autocast" is the reference's training
  mode (fp32 master weights and residual stream under bf16 autocast), with the block's RMSNorm
  passed in and, with ``valid`` < 1, the padding rows left out through ``unpad_indices``.
* ``experts`` ``scattermoe.mlp.GLUMLP`` on given routing (an expert-parallel share, or a
  caller with a router of its own). ``skew`` is the Zipf exponent of the experts' popularity.
* ``mlp``     ``scattermoe.mlp.MLP``: expert biases and GELU, through ``ParallelExperts``.
* ``shared``  ``modeling.expert_layer.ExpertMLP``: the dense SwiGLU expert.
* ``norm``    ``modeling.zRMSNorm.ZeroCenteredRMSNorm``.
* ``muon``    ``zmoe.muon.zeropower_via_newtonschulz5`` over a stack of expert weights' updates.

``train`` cases run forward and backward and return the output with every gradient.

Dimensions: d (hidden), E (routed experts), k (experts per token), f (expert width), fs (shared
expert width); the widths are those of the package's tests and benchmark and the reference's
default configuration (d = 512, f = 160, 32 routed + 2 shared experts, top-2).
"""

import math
import os
import sys

import torch
import torch.nn as nn
import torch.nn.functional as F

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PACKAGE = os.path.join(_ROOT, "architecture-zarelga-superposition_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

_BF16, _F32, _F64 = torch.bfloat16, torch.float32, torch.float64


# ------------------------------------------------------------------ the cases
def _layer(B, S, d, E, k, f, fs, mode, train, valid=1.0):
    return {"kind": "layer", "B": B, "S": S, "d": d, "E": E, "k": k, "f": f, "fs": fs, "mode": mode, "train": train,
            "valid": valid}


def _experts(T, d, E, k, f, dtype, train, skew):
    return {"kind": "experts", "T": T, "d": d, "E": E, "k": k, "f": f, "dtype": dtype, "train": train, "skew": skew}


def listed():
    cases = {
        # one decoding step of four sequences: latency, weight streaming of ~30 experts
        "layer_decode_4": _layer(4, 1, 2048, 128, 8, 768, 768, "bf16", False),
        # a prompt of ordinary, ragged length: ~126 rows an expert
        "layer_prefill_2011": _layer(1, 2011, 2048, 128, 8, 768, 1536, "bf16", False),
        # the reference's default configuration in its training mode, padded rows left out
        "layer_train_default": _layer(16, 512, 512, 32, 2, 160, 320, "autocast", True, 0.8),
        # the training step the package's benchmark runs
        "layer_train_32768": _layer(8, 4096, 2048, 128, 8, 768, 1536, "bf16", True),
        # a decoding batch with speculative tokens, or a short chunk: most experts get a few rows
        "experts_chunk_509": _experts(509, 2048, 128, 8, 768, "bf16", False, 0.0),
        # a large prefill on 64 narrow experts
        "experts_prefill_16384": _experts(16384, 1024, 64, 8, 512, "bf16", False, 0.3),
        # a quarter (expert-parallel share) of 256 experts of a 7168-wide model, skewed routing
        "experts_train_skewed": _experts(8192, 7168, 64, 2, 2048, "bf16", True, 1.1),
        # fp32 training of a small model
        "experts_train_fp32": _experts(2048, 256, 8, 2, 512, "f32", True, 0.3),
        # expert MLPs with biases at widths that are not whole 16-byte chunks
        "mlp_train_ragged": {"kind": "mlp", "T": 4001, "d": 510, "E": 16, "k": 2, "f": 1030, "train": True,
                             "skew": 0.3},
        # the dense expert on its own, a ragged number of rows
        "shared_train_8190": {"kind": "shared", "T": 8190, "d": 2048, "f": 1536, "train": True},
        # the norm in front of the layer
        "norm_train_16383": {"kind": "norm", "T": 16383, "d": 2048, "train": True},
        # the optimizer's orthogonalisation of one stack of 64 experts' updates
        "muon_64x1024x1024": {"kind": "muon", "E": 64, "m": 1024, "n": 1024, "steps": 5},
    }
    return [dict(c, name=name) for name, c in cases.items()]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


_WIDTHS = [(512, 32, 2, 160), (1024, 64, 8, 512), (2048, 128, 8, 768), (2048, 64, 4, 1024), (7168, 32, 2, 2048)]


_MOST_FLOPS = 9e12  # a drawn case costs no more than layer_train_32768


def draw(rng):
    """One more case of the listed ones' ranges."""
    case = _draw(rng)
    while work(case)["flops"] > _MOST_FLOPS:
        size = "S" if case["kind"] == "layer" else "T"
        case[size] = case[size] // 2 + 1
    return case


def _draw(rng):
    kind = rng.choice(["layer", "layer", "layer", "experts", "experts", "experts_f32", "mlp", "shared", "norm",
                       "muon"])
    d, E, k, f = rng.choice(_WIDTHS)
    skew = round(rng.uniform(0.0, 1.2), 2)
    train = rng.random() < 0.5
    if kind == "layer":
        fs = f * rng.choice([1, 2])
        if not train:
            T = _log(rng, 1, 16384)
            B = rng.choice([b for b in (1, 2, 4, 16, 64) if b <= T])
            return _layer(B, max(1, T // B), d, E, k, f, fs, "bf16", False)
        mode = rng.choice(["bf16", "autocast"])
        B, S = rng.choice([1, 2, 4, 8]), _log(rng, 64, 2048)
        valid = round(rng.uniform(0.5, 1.0), 2) if mode == "autocast" else 1.0
        return _layer(B, S, d, E, k, f, fs, mode, True, valid)
    if kind == "experts":
        return _experts(_log(rng, 64, 16384) if train else _log(rng, 1, 16384), d, E, k, f, "bf16", train, skew)
    if kind == "experts_f32":
        d, E, f = rng.choice([(256, 8, 512), (512, 32, 160), (384, 16, 640)])
        return _experts(_log(rng, 64, 8192), d, E, 2, f, "f32", train, skew)
    if kind == "mlp":
        return {"kind": "mlp", "T": _log(rng, 64, 8192), "d": rng.randrange(250, 1030), "E": rng.choice([8, 16, 32]),
                "k": rng.choice([1, 2, 4]), "f": rng.randrange(500, 2060), "train": train, "skew": skew}
    if kind == "shared":
        return {"kind": "shared", "T": _log(rng, 1, 16384), "d": d, "f": f * rng.choice([1, 2]), "train": train}
    if kind == "norm":
        return {"kind": "norm", "T": _log(rng, 1, 32768), "d": rng.choice([512, 1024, 2048, 4096, 7168]),
                "train": train}
    m, n = 8 * _log(rng, 12, 128), 8 * _log(rng, 12, 192)
    return {"kind": "muon", "E": _log(rng, 4, 64), "m": m, "n": n, "steps": 5}


# ------------------------------------------------------------------ inputs, from the seed alone
def _dev():
    return torch.device("cuda")


def _rand(seed):
    g = torch.Generator(device=_dev())
    g.manual_seed(seed)

    def normal(*shape, std=1.0, dtype=_F32):
        return torch.randn(*shape, device=_dev(), generator=g, dtype=dtype).mul_(std)

    return g, normal


def _routing(case, g):
    """k distinct experts a token, drawn by popularity rank ** -skew (Gumbel top-k over a random
    ranking), and L1-normalised weights, as a sigmoid router gives them."""
    T, E, k = case["T"], case["E"], case["k"]
    rank = torch.randperm(E, device=_dev(), generator=g).add_(1).float()
    u = torch.rand(T, E, device=_dev(), generator=g).clamp_(1e-9, 1 - 1e-7)
    idx = torch.topk(-torch.log(-torch.log(u)) - case["skew"] * torch.log(rank), k, dim=-1).indices
    p = torch.rand(T, k, device=_dev(), generator=g) * 0.5 + 0.4
    return idx, p / p.sum(-1, keepdim=True)


def _inputs(case, seed):
    g, normal = _rand(seed)
    kind = case["kind"]
    if kind == "layer":
        d, E, f, fs = (case[n] for n in ("d", "E", "f", "fs"))
        wt = _BF16 if case["mode"] == "bf16" else _F32
        std = d ** -0.5
        t = {"weights": {
            "gate.weight": normal(E, d, std=std, dtype=wt),
            "gate.expert_biases": normal(E, std=0.1),
            "shared_experts.gate_proj.weight": normal(fs, d, std=std, dtype=wt),
            "shared_experts.up_proj.weight": normal(fs, d, std=std, dtype=wt),
            "shared_experts.down_proj.weight": normal(d, fs, std=std, dtype=wt),
            "routed_experts.experts.weight": normal(E, 2 * f, d, std=std, dtype=wt),
            "routed_experts.output_experts.weight": normal(E, d, f, std=std, dtype=wt)}}
        B, S = case["B"], case["S"]
        t["x"] = normal(B, S, d, dtype=wt)
        t["rows"] = t["norm"] = None
        if case["mode"] == "autocast":
            t["norm"] = normal(d, std=0.1)
            if case["valid"] < 1:
                # whole documents of random length, right-padded: the flat rows that hold tokens
                lo = max(1, int(S * (2 * case["valid"] - 1)))
                lens = torch.randint(lo, S + 1, (B, 1), device=_dev(), generator=g)
                lens[0] = S
                t["rows"] = (torch.arange(S, device=_dev()) < lens).flatten().nonzero().flatten()
        t["dout"] = normal(B, S, d, dtype=_BF16) if case["train"] else None
    elif kind in ("experts", "mlp"):
        T, d, E, f = (case[n] for n in ("T", "d", "E", "f"))
        dt = _F32 if case.get("dtype") == "f32" else _BF16
        std = d ** -0.5
        width = 2 * f if kind == "experts" else f
        t = {"weights": {"experts.weight": normal(E, width, d, std=std, dtype=dt),
                         "output_experts.weight": normal(E, d, f, std=std, dtype=dt)}}
        if kind == "mlp":
            t["weights"]["experts.bias"] = normal(E, f, std=0.1, dtype=dt)
            t["weights"]["output_experts.bias"] = normal(E, d, std=0.1, dtype=dt)
        t["x"] = normal(T, d, dtype=dt)
        t["idx"], t["p"] = _routing(case, g)
        t["dout"] = normal(T, d, dtype=dt) if case["train"] else None
    elif kind == "shared":
        T, d, f = case["T"], case["d"], case["f"]
        std = d ** -0.5
        t = {"weights": {n + ".weight": normal(*s, std=std, dtype=_BF16)
                         for n, s in (("gate_proj", (f, d)), ("up_proj", (f, d)), ("down_proj", (d, f)))}}
        t["x"] = normal(T, d, dtype=_BF16)
        t["dout"] = normal(T, d, dtype=_BF16) if case["train"] else None
    elif kind == "norm":
        T, d = case["T"], case["d"]
        t = {"weights": {"weight": normal(d, std=0.1, dtype=_BF16)}, "x": normal(T, d, std=2.0, dtype=_BF16),
             "dout": normal(T, d, dtype=_BF16) if case["train"] else None}
    else:
        # a momentum-averaged gradient: noise on a few strong directions
        E, m, n = case["E"], case["m"], case["n"]
        low = torch.bmm(normal(E, m, 8), normal(E, 8, n))
        t = {"G": normal(E, m, n).add_(low, alpha=0.5)}
    return t


class _Config:
    def __init__(self, case):
        self.hidden_size = case["d"]
        self.intermediate_size = case["fs"]  # the shared expert's width; the routed experts take f below
        self.n_shared_experts = 1
        self.n_experts_per_token = case["k"]
        self.n_routed_experts = case["E"]
        self.initializer_range = case["d"] ** -0.5


def _module(case):
    kind = case["kind"]
    with torch.device("meta"):  # the weights come from _inputs
        if kind == "layer":
            from modeling.moe_layer import MoELayer
            from scattermoe.mlp import GLUMLP

            layer = MoELayer(_Config(case))
            layer.routed_experts = GLUMLP(case["d"], case["f"], case["E"], case["k"])
            return layer
        if kind == "experts":
            from scattermoe.mlp import GLUMLP

            return GLUMLP(case["d"], case["f"], case["E"], case["k"])
        if kind == "mlp":
            from scattermoe.mlp import MLP

            return MLP(case["d"], case["f"], case["E"], case["k"], bias=True, activation=nn.GELU())
        if kind == "shared":
            from modeling.expert_layer import ExpertMLP

            cfg = _Config(dict(case, fs=case["f"], k=1, E=1))
            return ExpertMLP(cfg)
        from modeling.zRMSNorm import ZeroCenteredRMSNorm

        return ZeroCenteredRMSNorm(case["d"])


def prepare(case, seed):
    """Inputs, and the module with its weights, as a training or serving loop holds them."""
    t = _inputs(case, seed)
    state = {"case": case, **{n: v for n, v in t.items() if n != "weights"}}
    if case["kind"] == "muon":
        return state
    m = _module(case)
    m.load_state_dict(t["weights"], assign=True)
    state["module"] = m.requires_grad_(case["train"])
    if case["kind"] == "layer":
        state["norm"] = None
        if t["norm"] is not None:
            from modeling.zRMSNorm import ZeroCenteredRMSNorm

            norm = ZeroCenteredRMSNorm(case["d"])
            norm.load_state_dict({"weight": t["norm"]}, assign=True)
            state["norm"] = norm.requires_grad_(case["train"])
    if case["train"]:
        state["x"].requires_grad_(True)
        if "p" in state:
            state["p"].requires_grad_(True)
    return state


# ------------------------------------------------------------------ one pass
def _forward(s):
    kind, m = s["case"]["kind"], s["module"]
    if kind == "layer":
        if s["case"]["mode"] == "autocast":
            with torch.autocast("cuda", dtype=_BF16):
                return m(s["x"], unpad_indices=s["rows"], norm=s["norm"])
        return m(s["x"])
    if kind in ("experts", "mlp"):
        return (m(s["x"], s["p"], s["idx"]),)
    return (m(s["x"]),)


def run(s):
    if s["case"]["kind"] == "muon":
        from zmoe.muon import zeropower_via_newtonschulz5

        return {"X": zeropower_via_newtonschulz5(s["G"], s["case"]["steps"])}
    if not s["case"]["train"]:
        with torch.no_grad():
            out = _forward(s)
        return {"out": out[0], **({"topk_idx": out[1]} if len(out) > 1 else {})}
    leaves = {"x": s["x"], **dict(s["module"].named_parameters())}
    if s.get("p") is not None:
        leaves["p"] = s["p"]
    if s.get("norm") is not None:
        leaves["norm.weight"] = s["norm"].weight
    for v in leaves.values():  # optimizer.zero_grad(set_to_none=True)
        v.grad = None
    out = _forward(s)
    out[0].backward(s["dout"])
    got = {"out": out[0].detach(), **{"d " + n: v.grad for n, v in leaves.items()}}
    if len(out) > 1:
        got["topk_idx"] = out[1]
    return got


# ------------------------------------------------------------------ what a pass cannot do without
def _tokens(case):
    if case["kind"] == "layer":
        return int(case["B"] * case["S"] * case["valid"])
    return case["T"]


def work(case):
    kind, train = case["kind"], case.get("train", False)
    if kind == "muon":
        E, m, n = case["E"], min(case["m"], case["n"]), max(case["m"], case["n"])
        return {"bytes": E * m * n * (4 + 2), "flops": case["steps"] * E * 2 * (2 * m * m * n + m * m * m)}
    T, d = _tokens(case), case["d"]
    if kind == "norm":
        return {"bytes": T * d * 2 * (4 if train else 2) + d * 2 * (2 if train else 1), "flops": T * d * (12 if train else 4)}
    act = 4 if case.get("dtype") == "f32" or case.get("mode") == "autocast" else 2
    weight = act
    flops = bytes_ = 0
    if kind in ("layer", "experts", "mlp"):
        R, E, f = T * case["k"], case["E"], case["f"]
        mats = 2 if kind == "mlp" else 3
        touched = E * (1 - (1 - 1 / E) ** R) if not train else E  # a training step writes every expert's grads
        flops += 2 * mats * R * d * f
        bytes_ += touched * mats * d * f * weight + R * (8 + 4)
    if kind == "layer":
        flops += 2 * T * d * case["E"] + 6 * T * d * case["fs"]
        bytes_ += (case["E"] + 3 * case["fs"]) * d * weight
    if kind == "shared":
        flops += 6 * T * d * case["f"]
        bytes_ += 3 * case["f"] * d * weight
    if train:
        # input and weight grads; the weights' grads written, dout read, dx written
        return {"bytes": 2 * bytes_ + 4 * T * d * act, "flops": 3 * flops}
    return {"bytes": bytes_ + 2 * T * d * act, "flops": flops}


def tolerance(case):
    """Measured against ``exact`` (about four times what the present code shows there), so that
    another order of the sums, and bf16 roundings at other places, stay inside."""
    if case["kind"] == "muon":
        return {"rel": 0.03}       # bf16 iteration: each step amplifies the last one's roundings
    if case.get("dtype") == "f32":
        return {"rel": 3e-6}
    if case["kind"] == "norm":
        return {"rel": 0.007}
    if case["kind"] == "layer":
        # a logit on a rounding boundary may choose another expert for its token
        return {"rel": 0.025, "max": 0.99, "differ": 0.01}
    return {"rel": 0.016}


# ------------------------------------------------------------------ the same in 64 bits
def _route64(x64, wg, bias, k):
    """The router on bf16 logits: probabilities rounded to bf16 choose (ties to the lowest
    expert), unrounded ones weigh."""
    logits = x64 @ wg.T
    with torch.no_grad():
        b = x64.to(_BF16).to(_F64) @ wg.to(_BF16).to(_F64).T
        score = torch.sigmoid(b.to(_F32).to(_BF16).to(_F64)).to(_F32).to(_BF16).to(_F32) + bias
        idx = torch.sort(score, dim=-1, descending=True, stable=True).indices[:, :k]
    p = torch.sigmoid(logits).gather(1, idx)
    return idx, p / p.sum(-1, keepdim=True)


def _experts64(x, idx, p, w):
    """sum_j p[t, j] * expert_{idx[t, j]}(x[t]), expert by expert."""
    W1, W2 = w["experts.weight"], w["output_experts.weight"]
    b1, b2 = w.get("experts.bias"), w.get("output_experts.bias")
    parts, rows = [], []
    for e in range(W1.shape[0]):
        t, j = (idx == e).nonzero(as_tuple=True)
        h = x.index_select(0, t) @ W1[e].T
        if b1 is None:
            up, gate = h.chunk(2, dim=-1)
            a = F.silu(gate) * up
        else:
            a = F.gelu(h + b1[e])
        y = a @ W2[e].T
        y = y if b2 is None else y + b2[e]
        parts.append(y * p[t, j].unsqueeze(1))
        rows.append(t)
    out = torch.zeros_like(x)
    return out.index_add(0, torch.cat(rows), torch.cat(parts))


def _norm64(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * (1 + w)


def _swiglu64(x, w):
    return (F.silu(x @ w["gate_proj.weight"].T) * (x @ w["up_proj.weight"].T)) @ w["down_proj.weight"].T


def exact(case, seed):
    t = _inputs(case, seed)
    if case["kind"] == "muon":
        X = t["G"].to(_F64)
        tall = case["m"] > case["n"]
        X = X.transpose(1, 2).contiguous() if tall else X
        X = X / (X.square().sum((1, 2), keepdim=True).sqrt() + 1e-7)
        for _ in range(case["steps"]):
            A = X @ X.transpose(1, 2).contiguous()
            X = 3.4445 * X + (-4.7750 * A + 2.0315 * (A @ A)) @ X
        return {"X": X.transpose(1, 2) if tall else X}
    train = case["train"]
    leaf = lambda v: v.to(_F64).requires_grad_(train and v.is_floating_point())  # noqa: E731
    w = {n: leaf(v) for n, v in t["weights"].items()}
    x = leaf(t["x"])
    leaves = {"x": x, **w}
    got = {}
    if case["kind"] == "layer":
        d = case["d"]
        bias = w.pop("gate.expert_biases").detach().to(_F32)
        leaves.pop("gate.expert_biases")
        flat = x.reshape(-1, d)
        if t["norm"] is not None:
            leaves["norm.weight"] = leaf(t["norm"])
            flat = _norm64(flat, leaves["norm.weight"])
        rows = t["rows"]
        inner = flat if rows is None else flat.index_select(0, rows)
        idx, p = _route64(inner, w["gate.weight"], bias, case["k"])
        sub = lambda pre: {n[len(pre):]: v for n, v in w.items() if n.startswith(pre)}  # noqa: E731
        out = _swiglu64(inner, sub("shared_experts.")) + _experts64(inner, idx, p, sub("routed_experts."))
        if rows is not None:
            out = torch.zeros_like(flat).index_copy(0, rows, out)
        out = out.view(x.shape)
        got["topk_idx"] = None
    elif case["kind"] in ("experts", "mlp"):
        p = leaf(t["p"])
        leaves["p"] = p
        out = _experts64(x, t["idx"], p, w)
    elif case["kind"] == "shared":
        out = _swiglu64(x, w)
    else:
        out = _norm64(x, w["weight"])
    got["out"] = out.detach()
    if train:
        grads = torch.autograd.grad(out, list(leaves.values()), t["dout"].to(_F64))
        got.update({"d " + n: v for n, v in zip(leaves, grads)})
    return got
