"""The MoE layer's measured cases: what programs call, over the range they call it at.

A case is a dict of plain values.  ``kind`` names the entry point:

* ``infer``   ``hanuman_amd.MoE`` without autograd: a decode step (``seq`` 1), a
  prompt, a long prefill; bfloat16 or float32 compute, sigmoid routing without
  drops (the reference's) or softmax routing with a capacity.
* ``train``   one training step of the layer: ``MoE`` under autograd, the
  gradients for the cotangents of its output and of the z and balance losses,
  and the in-place update that follows (so packed operands are made again in
  every step, as in a trainer's).
* ``layer``   ``hanuman_amd.layer.DeviceLayer.forward`` on packed weights: e4m3
  experts, and the load-skewed layer that routes from given logits.
* ``ragged``  ``hanuman_amd.moe.ragged_dispatch``: the functional form, which
  takes the float32 master weights in every call.
"""
import math

import torch

from hanuman_amd import MoE
from hanuman_amd.layer import DeviceLayer
from hanuman_amd.moe import ragged_dispatch
from hanuman_amd.workloads import Inputs, Workload, zipf_bias

Z_WEIGHT, BALANCE_WEIGHT = 1e-3, 1e-2   # weights of the aux losses in a training loss
LEARNING_RATE = 1e-7
ROUTER_STD = 0.02

# Layer shapes: the benchmark's bf16 layer, the reference's published MoE layer
# and a smaller generic one.
BF16_SHAPES = (
    dict(d_model=2048, experts=64, active=8, d_ff=1024),
    dict(d_model=1536, experts=80, active=8, d_ff=768),
    dict(d_model=1024, experts=16, active=2, d_ff=2048),
)
F32_SHAPES = (
    dict(d_model=256, experts=8, active=2, d_ff=512),
    dict(d_model=512, experts=16, active=4, d_ff=768),
)
FP8_SHAPES = (
    dict(d_model=4096, experts=32, active=4, d_ff=2048),
    dict(d_model=2048, experts=64, active=8, d_ff=1024),
)
SKEWED_SHAPE = dict(d_model=2048, experts=128, active=8, d_ff=768)


def _infer(batch, seq, shape, dtype="bf16", routing="sigmoid", capacity=0.0, shared=1, **more):
    return dict(kind="infer", batch=batch, seq=seq, dtype=dtype, routing=routing,
                capacity=capacity, shared=shared, **shape, **more)


def _train(batch, seq, shape, dtype="bf16", shared=1, **more):
    return dict(kind="train", batch=batch, seq=seq, dtype=dtype, routing="sigmoid", capacity=0.0,
                shared=shared, **shape, **more)


def _layer(tokens, shape, dtype, from_logits, **more):
    return dict(kind="layer", batch=1, seq=tokens, dtype=dtype, routing="softmax", capacity=1.25,
                shared=0, from_logits=from_logits, **shape, **more)


def _ragged(tokens, shape, **more):
    return dict(kind="ragged", batch=1, seq=tokens, dtype="bf16", routing="sigmoid", capacity=0.0,
                shared=0, **shape, **more)


def listed():
    return [
        # one sequence's decode step: one token, eight experts
        _infer(1, 1, BF16_SHAPES[0], name="decode_1"),
        # a serving batch's decode step: a few rows on nearly every expert
        _infer(48, 1, BF16_SHAPES[0], name="decode_48"),
        # one short prompt of odd length: some thirty rows an expert
        _infer(1, 333, BF16_SHAPES[1], name="prompt_333"),
        # a prefill batch at the reference's published layer
        _infer(4, 1024, BF16_SHAPES[1], name="prefill_4096"),
        # the benchmark's bf16 layer with its capacity, the largest prefill
        _infer(8, 2048, BF16_SHAPES[0], routing="softmax", capacity=1.25, name="prefill_16384"),
        # float32 compute on a few ragged prompts
        _infer(3, 257, F32_SHAPES[1], dtype="f32", name="prompt_771_f32"),
        # e4m3 experts: a serving batch, and the benchmark's e4m3 layer
        _layer(100, FP8_SHAPES[0], "fp8", False, name="fp8_100"),
        _layer(8192, FP8_SHAPES[0], "fp8", False, name="fp8_8192"),
        # many experts under a skewed load, with drops
        _layer(20000, SKEWED_SHAPE, "bf16", True, name="skewed_20000"),
        # training steps: the published layer in bf16, the small layer in float32
        _train(2, 1024, BF16_SHAPES[1], name="train_2048"),
        _train(4, 512, F32_SHAPES[0], dtype="f32", name="train_2048_f32"),
        # the functional form on master weights
        _ragged(1000, BF16_SHAPES[2], name="ragged_1000"),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    which = rng.choice(["decode", "prompt", "prompt", "prefill", "f32", "fp8", "fp8", "skewed",
                        "train", "train", "train_f32", "ragged"])
    if which == "decode":
        return _infer(_log_int(rng, 1, 256), 1, rng.choice(BF16_SHAPES),
                      shared=rng.choice([1, 1, 2]))
    if which == "prompt":
        return _infer(rng.randint(1, 3), _log_int(rng, 16, 1024), rng.choice(BF16_SHAPES),
                      shared=rng.choice([1, 1, 2]))
    if which == "prefill":
        routing = rng.choice(["sigmoid", "softmax"])
        return _infer(rng.randint(1, 8), _log_int(rng, 512, 2048), rng.choice(BF16_SHAPES),
                      routing=routing, capacity=1.25 if routing == "softmax" else 0.0)
    if which == "f32":
        return _infer(rng.randint(1, 4), _log_int(rng, 1, 512), rng.choice(F32_SHAPES), dtype="f32",
                      shared=rng.choice([1, 2]))
    if which == "fp8":
        return _layer(_log_int(rng, 16, 8192), rng.choice(FP8_SHAPES), "fp8", False)
    if which == "skewed":
        return _layer(_log_int(rng, 1000, 20000), SKEWED_SHAPE, "bf16", True)
    if which == "train":
        return _train(rng.randint(1, 4), _log_int(rng, 128, 1024), rng.choice(BF16_SHAPES[1:]))
    if which == "train_f32":
        return _train(rng.randint(1, 4), _log_int(rng, 32, 512), F32_SHAPES[0], dtype="f32",
                      shared=rng.choice([1, 2]))
    return _ragged(_log_int(rng, 16, 2048), BF16_SHAPES[2])


# ------------------------------------------------------------------ states --

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(g, shape, std=1.0):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).mul_(std)


_DT = {"bf16": torch.bfloat16, "f32": torch.float32}


def _module(case, seed):
    layer = MoE(case["d_model"], case["d_ff"], case["experts"], case["active"], case["shared"],
                ROUTER_STD, 2.5, _DT[case["dtype"]], seed, routing=case["routing"],
                capacity_factor=case["capacity"] or None)
    g = _generator(seed + 1)
    # a trained layer's balancing bias is small and not zero
    layer.bias.value.copy_(_normal(g, (case["experts"],), 0.01))
    x = _normal(g, (case["batch"], case["seq"], case["d_model"])).to(_DT[case["dtype"]])
    return layer, x, g


def _layer_inputs(case, seed):
    """The inputs of a ``layer`` case on the GPU: x, router or logits, weights."""
    g = _generator(seed)
    T, D, N, F = case["seq"], case["d_model"], case["experts"], case["d_ff"]
    x = _normal(g, (T, D)).to(torch.bfloat16).float()
    if case["from_logits"]:
        import numpy as np
        bias = torch.from_numpy(zipf_bias(N, np.random.default_rng(seed))).cuda()
        route = _normal(g, (T, N)) + bias
    else:
        route = _normal(g, (D, N), ROUTER_STD).to(torch.bfloat16).float()
    return (x, route, _normal(g, (N, D, F), 0.02), _normal(g, (N, D, F), 0.02),
            _normal(g, (N, F, D), 0.02))


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("infer", "train"):
        layer, x, g = _module(case, seed)
        if kind == "infer":
            with torch.no_grad():
                if case["dtype"] == "bf16":
                    # a served model has packed its weights; it does so in its first call
                    layer(x[:1, :1])
            return {"kind": kind, "layer": layer, "x": x}
        params = [p.value for n, p in layer.named_params().items() if n != "bias"]
        for p in params:
            p.requires_grad_(True)
        x.requires_grad_(True)
        return {"kind": kind, "layer": layer, "x": x, "params": params,
                "dy": _normal(g, (case["batch"], case["seq"], case["d_model"]), 1e-2),
                "dz": torch.tensor(Z_WEIGHT, device="cuda"),
                "dbal": torch.tensor(BALANCE_WEIGHT, device="cuda")}
    if kind == "layer":
        x, route, wg, wu, wd = (t.cpu().numpy() for t in _layer_inputs(case, seed))
        wl = Workload("case", tokens=case["seq"], d_model=case["d_model"], n_experts=case["experts"],
                      top_k=case["active"], d_ff=case["d_ff"], capacity_factor=case["capacity"],
                      router_from_logits=case["from_logits"], expert_dtype=case["dtype"],
                      router_w_dtype="bf16" if case["dtype"] == "fp8" else "f32",
                      out_dtype="bf16" if case["dtype"] == "fp8" else "f32")
        inp = Inputs(wl, x, w_gate=wg, w_up=wu, w_down=wd)
        if case["from_logits"]:
            inp.logits = route
        else:
            inp.router = route
        return {"kind": kind, "layer": DeviceLayer(inp)}
    return {"kind": kind, **_ragged_inputs(case, seed)}


def _ragged_inputs(case, seed):
    g = _generator(seed)
    T, D, N, F, K = (case[k] for k in ("seq", "d_model", "experts", "d_ff", "active"))
    std = D ** -0.5
    top = torch.rand((T, N), generator=g, device="cuda").topk(K, dim=1).indices.to(torch.int32)
    w = torch.rand((T, K), generator=g, device="cuda") + 0.1
    return {"x": _normal(g, (T, D)).to(torch.bfloat16), "top_idx": top.contiguous(),
            "weights": w / w.sum(dim=1, keepdim=True), "w_gate": _normal(g, (N, D, F), std),
            "w_up": _normal(g, (N, D, F), std), "w_down": _normal(g, (N, F, D), std)}


def run(state):
    kind = state["kind"]
    if kind == "infer":
        with torch.no_grad():
            out, aux = state["layer"](state["x"])
        return {"out": out, **aux}
    if kind == "train":
        params = state["params"]
        out, aux = state["layer"](state["x"])
        grads = torch.autograd.grad((out, aux["router_z_loss"], aux["balance_loss"]),
                                    [state["x"], *params],
                                    (state["dy"], state["dz"], state["dbal"]))
        with torch.no_grad():
            torch._foreach_add_(params, list(grads[1:]), alpha=-LEARNING_RATE)
        return {"out": out.detach(), "grads": list(grads),
                "losses": [aux["router_z_loss"].detach(), aux["balance_loss"].detach()]}
    if kind == "layer":
        r = state["layer"].forward()
        return {"out": r["out"], "gates": r["gates"], "top_idx": r["top_idx"]}
    return ragged_dispatch(state["x"], state["top_idx"], state["weights"], state["w_gate"],
                           state["w_up"], state["w_down"], torch.bfloat16)


# ------------------------------------------------------------ what it costs --

def work(case):
    T = case["batch"] * case["seq"]
    D, N, F, K = (case[k] for k in ("d_model", "experts", "d_ff", "active"))
    rows = T * K
    if case["capacity"]:
        rows = min(rows, N * math.ceil(case["capacity"] * rows / N))
    touched = N * (1.0 - (1.0 - K / N) ** T)   # experts with a row, on average
    expert = 3 * D * F
    shared = case["shared"] * expert
    flops = 6.0 * D * F * (rows + case["shared"] * T) + (2.0 * T * D * N if case["kind"] != "ragged"
                                                         and not case.get("from_logits") else 0.0)
    act = 4 if case["dtype"] == "f32" else 2
    out = 2 if case["dtype"] == "fp8" else 4
    size = {"bf16": 2, "fp8": 1, "f32": 4}[case["dtype"]]
    if case["kind"] == "train":
        flops *= 3.0
        weights = N * expert + shared + D * N
        # masters read once, gradients written, the masters updated; x, dy, dx, out
        return {"bytes": weights * 12.0 + T * D * (2 * act + 8), "flops": flops}
    if case["kind"] == "ragged":
        return {"bytes": touched * expert * 4.0 + T * D * (act + 4) + T * K * 8, "flops": flops}
    route = T * N * 4 if case.get("from_logits") else D * N * (2 if case["dtype"] == "fp8" else 4)
    return {"bytes": (touched * expert + shared) * size + T * D * (act + out) + route, "flops": flops}


def tolerance(case):
    if case["dtype"] == "f32":
        return {"rel": 1e-5, "max": 1e-3}
    if case["dtype"] == "fp8":
        return {"rel": 1e-2, "max": 0.2}
    return {"rel": 1e-2, "max": 0.2}


# ------------------------------------------------------------------ 64 bits --
# The layer in float64 torch.  Weights and activations enter with the values
# the compute dtype gives them (bfloat16-rounded masters; nothing between is
# rounded); the selection is made on float32 logits, as the layer defines it.

def _select(logits, bias, K, routing):
    """(top_idx, gates): lower index first on equal keys."""
    key = logits if routing == "softmax" else torch.sigmoid(logits) + bias
    idx = torch.sort(key.float(), dim=1, descending=True, stable=True).indices[:, :K]
    return idx


def _experts(x, idx, gates, N, cap, weights):
    """sum over the kept slots of gate * SwiGLU_e(x); differentiable."""
    T, K = idx.shape
    out = torch.zeros((T, weights(0)[2].shape[1]), dtype=x.dtype, device=x.device)
    flat = idx.reshape(-1)
    for e in range(N):
        slots = (flat == e).nonzero().reshape(-1)[:cap]
        if not len(slots):
            continue
        tok = slots // K
        wg, wu, wd = weights(e)
        xe = x[tok]
        ye = (torch.nn.functional.silu(xe @ wg) * (xe @ wu)) @ wd
        out = out.index_add(0, tok, ye * gates.reshape(-1)[slots].unsqueeze(1))
    return out


def _module_exact(case, x, router, bias, wg, wu, wd, swg, swu, swd, rsf=2.5):
    """(out, z, balance, entropy, counts) of the module in float64."""
    B, S, N, K = case["batch"], case["seq"], case["experts"], case["active"]
    T = B * S
    x2 = x.reshape(T, -1)
    logits = x2 @ router
    idx = _select(logits.detach().float().double(), bias, K, case["routing"])
    scores = torch.sigmoid(logits)
    if case["routing"] == "softmax":
        gates = torch.softmax(torch.gather(logits, 1, idx), dim=1)
    else:
        sel = torch.gather(scores, 1, idx)
        gates = sel / (sel.sum(dim=1, keepdim=True) + 1e-9) * rsf
    cap = math.ceil(case["capacity"] * T * K / N) if case["capacity"] else T * K
    out = _experts(x2, idx, gates, N, cap, lambda e: (wg[e], wu[e], wd[e]))
    n = case["shared"]
    if n == 1:
        swg, swu, swd = swg.unsqueeze(0), swu.unsqueeze(0), swd.unsqueeze(0)
    for i in range(n):
        out = out + ((torch.nn.functional.silu(x2 @ swg[i]) * (x2 @ swu[i])) @ swd[i]) / n
    lse = torch.logsumexp(logits, dim=1)
    counts = torch.zeros((B, N), dtype=torch.float64, device=x.device)
    counts.scatter_add_(1, idx.reshape(B, S * K),
                        torch.ones((B, S * K), dtype=torch.float64, device=x.device))
    probs = scores / (scores.sum(dim=1, keepdim=True) + 1e-9)
    balance = (N * (counts / (S * K) * probs.reshape(B, S, N).mean(dim=1)).sum(dim=1)).mean()
    entropy = -(probs * torch.log(probs + 1e-9)).sum(dim=1).mean()
    return out.reshape(B, S, -1), (lse * lse).mean(), balance, entropy, counts.sum(dim=0)


def exact(case, seed):
    kind = case["kind"]
    round_w = (lambda t: t.double()) if case["dtype"] == "f32" else (
        lambda t: t.to(torch.bfloat16).double())
    if kind in ("infer", "train"):
        layer, x, g = _module(case, seed)
        p = {n: v.value for n, v in layer.named_params().items()}
        names = ("expert_w_gate", "expert_w_up", "expert_w_down", "shared_w_gate", "shared_w_up",
                 "shared_w_down")
        weights = [round_w(p[n]) for n in names]
        args = [x.double(), p["router"].double(), p["bias"].double(), *weights]
        if kind == "infer":
            with torch.no_grad():
                out, z, bal, ent, counts = _module_exact(case, *args)
            return {"out": out, "router_z_loss": z, "balance_loss": bal, "mean_entropy": ent,
                    "expert_counts": counts}
        dy = _normal(g, (case["batch"], case["seq"], case["d_model"]), 1e-2).double()
        wanted = [args[0], args[1], *weights]
        for t in wanted:
            t.requires_grad_(True)
        out, z, bal, _, _ = _module_exact(case, *args)
        loss = (out * dy).sum() + Z_WEIGHT * z + BALANCE_WEIGHT * bal
        grads = torch.autograd.grad(loss, wanted)
        return {"out": out.detach(), "grads": list(grads), "losses": [z.detach(), bal.detach()]}
    if kind == "layer":
        x, route, wg, wu, wd = (t.double() for t in _layer_inputs(case, seed))
        logits = route if case["from_logits"] else x @ route
        N, K, T = case["experts"], case["active"], case["seq"]
        idx = _select(logits.float().double(), None, K, "softmax")
        gates = torch.softmax(torch.gather(logits, 1, idx), dim=1)
        cap = math.ceil(case["capacity"] * T * K / N)
        if case["dtype"] == "fp8":
            def q(t):   # a column's e4m3 codes, as the layer's weights hold them
                s = t.abs().amax(dim=0, keepdim=True) / 448.0
                s = torch.where(s == 0, torch.ones_like(s), s)
                return (t / s).float().to(torch.float8_e4m3fn).double() * s
        else:
            q = round_w
        out = _experts(x, idx, gates, N, cap, lambda e: (q(wg[e]), q(wu[e]), q(wd[e])))
        return {"out": out, "gates": gates, "top_idx": None}
    s = _ragged_inputs(case, seed)
    N = case["experts"]
    return _experts(s["x"].double(), s["top_idx"].long(), s["weights"].double(), N,
                    case["seq"] * case["active"],
                    lambda e: (round_w(s["w_gate"][e]), round_w(s["w_up"][e]), round_w(s["w_down"][e])))
