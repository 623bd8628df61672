"""The workloads that this package's speed is measured on, through its public entry points.

Five kinds of case, each a dict of plain values:

  layer    moe_amd.layer.moe_layer: gating linear, router, experts; forward only (serving,
           evaluation) or forward + backward (training), softmax or sigmoid router, bf16 or
           fp32, per-layer experts or a shared bank whose gradient adds into ``main_grad``
  experts  moe_amd.experts_forward on a given routing (the transformers plug-in's call)
  router   MI355XDeepSeekRouter, forward + backward, with selection counts
  aux      the load-balancing losses over all layers' router outputs, with their gradients

``listed()`` holds the sizes a user of the package runs (the benchmark's five layers among
them), ``draw()`` others of the same ranges.  Inputs follow the benchmark's distributions:
hidden states and output gradients N(0, 1), weights N(0, 0.02).
"""
from __future__ import annotations

import math
from types import SimpleNamespace

import torch

from moe_amd import MI355XDeepSeekRouter, experts_forward
from moe_amd.balancing import load_balancing_loss_func, seq_load_balancing_loss_func
from moe_amd.layer import moe_layer

DEV = "cuda"

LAYER = dict(kind="layer", dtype="bf16", router="softmax", train=False, bank=False, skew=0.0,
             bias_range=0.0)
EXPERTS = dict(kind="experts", dtype="bf16", train=False, skew=0.0)


def listed():
    big = dict(H=2048, E=128, K=8, I=768)
    xs = dict(H=1024, K=4, I=768)
    return [
        # a decode step of a small serving batch: weight streaming, launches and host time
        dict(LAYER, name="decode_4", T=4, **big),
        # a ragged prefill chunk (chunked prefill, speculative verification)
        dict(LAYER, name="chunk_333", T=333, **big),
        # one long prompt's prefill, of an odd length
        dict(LAYER, name="prefill_4095", T=4095, **big),
        # the XS layer in fp32, forward: evaluation at the reference's own precision
        dict(LAYER, name="xs_f32_forward", T=2048, E=16, dtype="f32", **xs),
        # the fp32 experts of a training step under bf16 autocast (parameters stay fp32 there)
        dict(EXPERTS, name="f32_train", T=8192, E=16, dtype="f32", train=True, **xs),
        # a small research model's expert layer, odd token count, skewed routing
        dict(EXPERTS, name="small_train", T=1531, H=512, E=64, K=6, I=256, train=True, skew=1.0),
        # a training call on the XS model's shared bank, gradients added into main_grad
        dict(LAYER, name="xs_global_train", T=16384, E=128, train=True, bank=True, **xs),
        # a training step of the M layer with Zipf-skewed routing
        dict(LAYER, name="m_skew_train", T=32768, train=True, skew=2.0, **big),
        # a training step of the L layer: the largest
        dict(LAYER, name="l_train", T=65536, train=True, **big),
        # a training call on the 1792-expert bank: sigmoid router with expert bias, main_grad
        dict(LAYER, name="retrofit_train", T=16384, H=2048, E=1792, K=8, I=768, train=True,
             router="sigmoid", bias_range=0.5, bank=True),
        # the DeepSeek router of a training step: group-limited selection, counts, gradients
        dict(kind="router", name="deepseek_router", T=32768, H=2048, E=128, K=8, groups=8,
             group_topk=4, scaling=2.5),
        # the sequence-wise balancing loss over the layers of a model, with gradients
        dict(kind="aux", name="seq_aux_loss", loss="seq", layers=16, B=8, S=2048, E=128, K=4),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "prefill", "train", "experts", "f32_forward", "f32_train",
                       "router", "aux"])
    big = [dict(H=2048, E=128, K=8, I=768), dict(H=1024, E=128, K=4, I=768),
           dict(H=2048, E=64, K=8, I=768)]
    small = [dict(H=512, E=64, K=8, I=256), dict(H=320, E=24, K=3, I=320),
             dict(H=1024, E=16, K=4, I=768), dict(H=512, E=64, K=6, I=256)]
    if kind == "decode":
        router = rng.choice(["softmax", "softmax", "sigmoid"])
        return dict(LAYER, T=_log_int(rng, 1, 96), router=router,
                    bias_range=0.1 if router == "sigmoid" else 0.0, **rng.choice(big + small[:2]))
    if kind == "prefill":
        return dict(LAYER, T=_log_int(rng, 97, 16384), skew=rng.choice([0.0, 2.0]),
                    **rng.choice(big))
    if kind == "train":
        return dict(LAYER, T=_log_int(rng, 512, 32768), train=True, bank=rng.random() < 0.3,
                    skew=rng.choice([0.0, 0.0, 2.0]), **rng.choice(big))
    if kind == "experts":
        return dict(EXPERTS, T=_log_int(rng, 64, 8192), train=rng.random() < 0.7,
                    skew=rng.choice([0.0, 1.0]), **rng.choice(small))
    if kind == "f32_forward":
        return dict(LAYER, T=_log_int(rng, 16, 4096), dtype="f32", **rng.choice(small))
    if kind == "f32_train":
        return dict(EXPERTS, T=_log_int(rng, 256, 8192), dtype="f32", train=True,
                    skew=rng.choice([0.0, 1.0]), **rng.choice(small + big[1:2]))
    if kind == "router":
        E, K, groups, keep = rng.choice([(128, 8, 8, 4), (64, 8, 8, 4), (128, 8, 0, 0),
                                         (64, 6, 0, 0), (256, 8, 8, 4)])
        return dict(kind="router", T=_log_int(rng, 256, 65536), H=rng.choice([512, 1024, 2048]),
                    E=E, K=K, groups=groups, group_topk=keep, scaling=rng.choice([0.0, 2.5]))
    loss = rng.choice(["seq", "switch"])
    E, K = rng.choice([(128, 8), (128, 4), (64, 6)])
    return dict(kind="aux", loss=loss, layers=rng.randint(4, 24), B=rng.choice([1, 2, 4, 8]),
                S=_log_int(rng, 200, 2048), E=E, K=K)


# ------------------------------------------------------------------ inputs

def _dtype(case):
    return torch.float32 if case["dtype"] == "f32" else torch.bfloat16


def _normal(g, shape, std, dtype):
    return torch.empty(shape, device=DEV, dtype=dtype).normal_(0.0, std, generator=g)


def _zipf(g, E, scale):
    """Per-expert logit offset of a skewed routing: scale * rank^-1.1, ranks shuffled."""
    rank = torch.randperm(E, generator=g, device=DEV).to(torch.float32) + 1.0
    return scale * rank.pow(-1.1)


def prepare(case, seed):
    g = torch.Generator(device=DEV).manual_seed(int(seed))
    kind = case["kind"]
    if kind == "router":
        T, H, E = case["T"], case["H"], case["E"]
        router = MI355XDeepSeekRouter(SimpleNamespace(
            num_experts_per_tok=case["K"], num_experts=E, norm_topk_prob=True, hidden_size=H,
            topk_scaling_factor=case["scaling"] or None, num_groups=case["groups"] or None,
            group_topk=case["group_topk"] or None)).to(DEV)
        router.weight = torch.nn.Parameter(_normal(g, (E, H), 0.02, torch.bfloat16))
        with torch.no_grad():
            router.expert_bias.uniform_(-0.02, 0.02, generator=g)
        return dict(case=case, router=router,
                    x=_normal(g, (T, H), 1.0, torch.bfloat16).requires_grad_(True),
                    d_w=_normal(g, (T, case["K"]), 1.0, torch.bfloat16),
                    d_scores=_normal(g, (T, E), 0.01, torch.float32))
    if kind == "aux":
        T, E, K = case["B"] * case["S"], case["E"], case["K"]
        layers, sel = [], []
        for _ in range(case["layers"]):
            logits = torch.randn(T, E, generator=g, device=DEV)
            p = torch.softmax(logits, -1) if case["loss"] == "switch" else torch.sigmoid(logits)
            sel.append(p.topk(K, dim=-1).indices)
            layers.append(p.requires_grad_(True))
        return dict(case=case, layers=tuple(layers), selected=tuple(sel))
    T, H, E, K, I = (case[k] for k in ("T", "H", "E", "K", "I"))
    dt = _dtype(case)
    s = dict(case=case, x=_normal(g, (T, H), 1.0, dt), w1=_normal(g, (E, 2 * I, H), 0.02, dt),
             w2=_normal(g, (E, H, I), 0.02, dt), wr=None, offset=None, bias=None)
    if kind == "layer":
        s["wr"] = _normal(g, (E, H), 0.02, dt)
        if case["skew"]:
            s["offset"] = _zipf(g, E, case["skew"])
        if case["bias_range"]:
            s["bias"] = (torch.rand(E, generator=g, device=DEV) * 2 - 1) * case["bias_range"]
    else:
        logits = torch.randn(T, E, generator=g, device=DEV)
        if case["skew"]:
            logits = logits + _zipf(g, E, case["skew"] * 4)
        w, s["idx"] = torch.softmax(logits, -1).topk(K, dim=-1)
        s["w"] = w / w.sum(-1, keepdim=True)
    if case["train"]:
        s["dout"] = _normal(g, (T, H), 1.0, dt)
        for k in ("x", "w1", "w2", "wr" if kind == "layer" else "w"):
            s[k].requires_grad_(True)
        if case.get("bank"):
            s["w1"].main_grad = torch.zeros_like(s["w1"], requires_grad=False)
            s["w2"].main_grad = torch.zeros_like(s["w2"], requires_grad=False)
    return s


# --------------------------------------------------------------- one pass

def _experts_grads(s, case):
    if case.get("bank"):
        return {"d_gate_up": s["w1"].main_grad, "d_down": s["w2"].main_grad}
    return {"d_gate_up": s["w1"].grad, "d_down": s["w2"].grad}


def run(state):
    s, case = state, state["case"]
    kind = case["kind"]
    if kind == "router":
        r = s["router"]
        r.local_tokens_per_expert.zero_()
        s["x"].grad = r.weight.grad = None
        scores, w, idx = r(s["x"])
        torch.autograd.backward([scores, w], [s["d_scores"], s["d_w"]])
        return {"scores": scores, "weights": w, "index": idx,
                "counts": r.local_tokens_per_expert, "d_x": s["x"].grad,
                "d_weight": r.weight.grad}
    if kind == "aux":
        for p in s["layers"]:
            p.grad = None
        if case["loss"] == "seq":
            loss = seq_load_balancing_loss_func(s["layers"], case["E"], case["K"], case["B"],
                                                s["selected"])
        else:
            loss = load_balancing_loss_func(s["layers"], case["E"], case["K"])
        loss.backward()
        return {"loss": loss, "grads": [p.grad for p in s["layers"]]}
    if case["train"]:
        for k in ("x", "w1", "w2", "wr", "w"):
            if s.get(k) is not None:
                s[k].grad = None
        if case.get("bank"):  # one micro-batch per optimizer step: the bank's gradient restarts
            s["w1"].main_grad.zero_()
            s["w2"].main_grad.zero_()
    if kind == "experts":
        with torch.set_grad_enabled(case["train"]):
            out = experts_forward(s["x"], s["idx"], s["w"], s["w1"], s["w2"])
        if not case["train"]:
            return {"out": out}
        out.backward(s["dout"])
        return {"out": out, "d_x": s["x"].grad, "d_w": s["w"].grad, **_experts_grads(s, case)}
    with torch.set_grad_enabled(case["train"]):
        out, probs, w, idx = moe_layer(s["x"], s["wr"], s["w1"], s["w2"], case["K"],
                                       router=case["router"], logit_offset=s["offset"],
                                       expert_bias=s["bias"])
    res = {"out": out, "probs": probs, "weights": w, "index": idx}
    if case["train"]:
        out.backward(s["dout"])
        res.update(d_x=s["x"].grad, d_router=s["wr"].grad, **_experts_grads(s, case))
    return res


# ------------------------------------------------------------ work, error

def _touched(case):
    """Experts that get at least one token: all of them at training sizes, K*T distinct
    draws at decode sizes, about a fifth under the wide expert bias."""
    E = case["E"] * (0.2 if case.get("bias_range", 0.0) >= 0.5 else 1.0)
    return E * (1.0 - (1.0 - case["K"] / E) ** case["T"]) if case["K"] < E else E


def work(case):
    kind = case["kind"]
    if kind == "aux":
        n = case["layers"] * case["B"] * case["S"]
        return {"bytes": n * case["E"] * 8.0 + n * case["K"] * 8.0, "flops": n * case["E"] * 8.0}
    T, H, E, K = (case[k] for k in ("T", "H", "E", "K"))
    if kind == "router":
        return {"bytes": 2.0 * 2 * T * H + 2.0 * 2 * E * H + 4.0 * 2 * T * E + T * K * 12.0,
                "flops": 6.0 * T * H * E}
    I, b = case["I"], 4.0 if case["dtype"] == "f32" else 2.0
    bank = 3.0 * H * I * b
    train = case["train"]
    nbytes = 2.0 * T * H * b + _touched(case) * bank
    flops = (18.0 if train else 6.0) * T * K * H * I
    if kind == "layer":
        nbytes += E * H * b + T * E * 4.0
        flops += (6.0 if train else 2.0) * T * H * E
    nbytes += T * K * 12.0
    if train:
        nbytes += 2.0 * T * H * b + E * bank
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # about four times what each kind differs from exact() by
    if case["kind"] in ("layer", "experts"):
        # bf16: one rounding per tensor of the chain (0.0049); fp32: summation order (1.2e-6)
        return {"rel": 2e-2} if case["dtype"] == "bf16" else {"rel": 5e-6}
    if case["kind"] == "router":
        return {"rel": 8e-3}  # bf16 gradients and weights (0.0018)
    return {"rel": 4e-6}  # fp32 gradients (5e-7, cancellation at balanced routing)


# ------------------------------------------------------- 64-bit reference

def _rank(values, K):
    """Top-K ids, value descending, lower id first on equal values."""
    return torch.sort(values, dim=-1, descending=True, stable=True).indices[:, :K]


def _experts64(s, case, idx, w):
    """The expert layer and its gradients in fp64, expert by expert.  Weight gradients of
    banks over 2^31 values are kept in fp32 (their bf16 counterparts carry 8 bits)."""
    x, w1, w2 = s["x"].detach(), s["w1"].detach(), s["w2"].detach()
    T, H = x.shape
    E, I, K = w1.shape[0], w2.shape[2], idx.shape[1]
    x64, w64 = x.double(), w.double()
    res = {"out": torch.zeros(T, H, dtype=torch.float64, device=DEV)}
    train = case["train"]
    if train:
        keep = torch.float32 if E * H * I >= 1 << 30 else torch.float64
        do = s["dout"].double()
        res["d_x"] = torch.zeros_like(res["out"])
        res["d_w"] = torch.zeros(T * K, dtype=torch.float64, device=DEV)
        res["d_gate_up"] = torch.zeros(w1.shape, dtype=keep, device=DEV)
        res["d_down"] = torch.zeros(w2.shape, dtype=keep, device=DEV)
    flat = idx.reshape(-1)
    order = torch.sort(flat, stable=True).indices
    counts = torch.bincount(flat, minlength=E).tolist()
    at = 0
    for e, n in enumerate(counts):
        if not n:
            continue
        src = order[at:at + n]
        at += n
        t, wk = src // K, w64.reshape(-1)[src][:, None]
        h, a1, a2 = x64[t], w1[e].double(), w2[e].double()
        g, u = (h @ a1.T).split(I, dim=1)
        sg = torch.sigmoid(g)
        act = g * sg * u
        y = act @ a2.T
        res["out"].index_add_(0, t, y * wk)
        if train:
            d = do[t]
            res["d_w"][src] = (d * y).sum(-1)
            dy = d * wk
            da = dy @ a2
            res["d_down"][e] = (dy.T @ act).to(keep)
            dgu = torch.cat([da * u * sg * (1 + g * (1 - sg)), da * g * sg], dim=1)
            res["d_gate_up"][e] = (dgu.T @ h).to(keep)
            res["d_x"].index_add_(0, t, dgu @ a1)
    if train:
        res["d_w"] = res["d_w"].reshape(T, K)
    return res


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind == "aux":
        T, E, K, B = case["B"] * case["S"], case["E"], case["K"], case["B"]
        ps = [p.detach().double().requires_grad_(True) for p in s["layers"]]
        if case["loss"] == "seq":
            total = 0.0
            for p, sel in zip(ps, s["selected"]):
                n = p / (p.sum(-1, keepdim=True) + 1e-20)
                f = torch.zeros(T, E, dtype=torch.float64, device=DEV).scatter_(1, sel, 1.0)
                f = f.reshape(B, -1, E).sum(1) * (E / (K * case["S"]))
                total = total + (f * n.reshape(B, -1, E).mean(1)).sum(-1).mean()
            loss = total / len(ps)
        else:
            f = sum(torch.zeros_like(p).scatter_(1, _rank(q.detach(), K), 1.0).sum(0)
                    for p, q in zip(ps, s["layers"])) / (T * len(ps))
            loss = (f.detach() * sum(p.sum(0) for p in ps) / (T * len(ps))).sum() * E
        loss.backward()
        return {"loss": loss.detach(), "grads": [p.grad for p in ps]}
    if kind == "experts":
        return _experts64(s, case, s["idx"], s["w"].detach())
    x, K, E = s["x"].detach(), case["K"], case["E"]
    wr = (s["router"].weight if kind == "router" else s["wr"]).detach()
    sigmoid = kind == "router" or case["router"] == "sigmoid"
    # the logits are part of the definition: the routing is decided on the gating linear as
    # torch computes it, in fp32 for the sigmoid router
    logits = (torch.nn.functional.linear(x.float(), wr.float()) if sigmoid
              else torch.nn.functional.linear(x, wr))
    train = kind == "router" or case["train"]
    l64 = logits.double().requires_grad_(train)
    scaling = 1.0
    if sigmoid:
        bias = s["router"].expert_bias if kind == "router" else s["bias"]
        ranked = torch.sigmoid(logits) + (bias if bias is not None else 0.0)
        if kind == "router":
            scaling = case["scaling"] or 1.0
            if case["groups"]:
                G, keep = case["groups"], case["group_topk"]
                by = ranked.reshape(-1, G, E // G)
                score = by.topk(K // keep, dim=-1).values.sum(-1)
                mask = torch.zeros_like(score).scatter_(1, _rank(score, keep), 1.0)
                ranked = by.masked_fill(mask[..., None] == 0, float("-inf")).reshape(-1, E)
        probs = torch.sigmoid(l64)
    else:
        ranked = logits.float() + (s["offset"] if s["offset"] is not None else 0.0)
        probs = torch.softmax(l64 + (s["offset"].double() if s["offset"] is not None else 0.0), -1)
    idx = _rank(ranked, K)
    w = probs.gather(1, idx)
    w = w / w.sum(-1, keepdim=True) * scaling
    if kind == "router":
        torch.autograd.backward([probs, w], [s["d_scores"].double(), s["d_w"].double()])
        return {"scores": probs.detach(), "weights": w.detach(), "index": None,
                "counts": torch.bincount(idx.reshape(-1), minlength=E).double(),
                "d_x": l64.grad @ wr.double(), "d_weight": l64.grad.T @ x.double()}
    res = _experts64(s, case, idx, w.detach())
    out = {"out": res["out"], "probs": probs.detach(), "weights": w.detach(), "index": None}
    if train:
        w.backward(res["d_w"])
        out.update(d_x=res["d_x"] + l64.grad @ wr.double(), d_router=l64.grad.T @ x.double(),
                   d_gate_up=res["d_gate_up"], d_down=res["d_down"])
    return out
