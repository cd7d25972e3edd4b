"""The work a serving engine has this library do, as cases to time and to check.

Experts are synthetic GGUF blobs (gate || up || down, whole blocks of 32
weights with one f16 scale each) with the value ranges of the benchmark:
Q4_0 nibbles uniform with d ~ U(0.005, 0.02), Q8_0 int8 uniform in
[-127, 127] with d ~ U(0.002, 0.01).  Hidden states are f32 N(0, 1).
Routing is top-k of N(0, 1) logits plus the log of a Zipf popularity, with
softmax weights over the chosen experts.  All of it is made on the GPU from
the seed with torch alone, so `exact` reads the same bytes.
"""
from __future__ import annotations

import importlib
import math

import torch

mer = importlib.import_module("micro-expert-router-ssd-streamed-moe-mer_amd")
routing = importlib.import_module("micro-expert-router-ssd-streamed-moe-mer_amd.routing")

DEV = "cuda"
BLOCK_BYTES = {"q4": 18, "q8": 34}
DTYPES = {"q4": mer.WeightDtype.Q4_0, "q8": mer.WeightDtype.Q8_0}


# ---- cases ---------------------------------------------------------------

def listed():
    return [
        # One decode step of Mixtral-8x7B: every layer's routed experts in
        # one call (the benchmark's headline workload).
        dict(name="stack_mixtral_q4", kind="stack", dtype="q4", layers=32, experts=8, top_k=2, tokens=1,
             d_model=4096, d_ff=14336, zipf=0.0),
        # The same for Qwen3-30B-A3B: many small experts, top-8.
        dict(name="stack_qwen3_q8", kind="stack", dtype="q8", layers=48, experts=128, top_k=8, tokens=1,
             d_model=2048, d_ff=768, zipf=0.0),
        # One layer of one decode step in the engine's default Q4_0
        # arithmetic (Q8_0 activations): the engine's own call pattern.
        dict(name="layer_mixtral_q4_qmm", kind="layer", dtype="q4", qmm=True, experts=8, top_k=2, tokens=1,
             d_model=4096, d_ff=14336, zipf=0.0),
        # A small decode batch (four sequences), DeepSeek-V3 experts.
        dict(name="layer_deepseek_q4_b4", kind="layer", dtype="q4", qmm=False, experts=256, top_k=8, tokens=4,
             d_model=7168, d_ff=2048, zipf=1.0),
        # One routed expert on one hidden state: the smallest call, and the
        # one parallel expert workers make.
        dict(name="expert_qwen3_q8", kind="expert", dtype="q8", qmm=False, d_model=2048, d_ff=768),
        # The GPU backend's f16 batch of eight experts on one hidden state.
        dict(name="views_qwen3_q4", kind="views", dtype="q4", experts=128, n=8, d_model=2048, d_ff=768),
        # A layer whose experts come and go between host RAM and a small VRAM
        # slot cache: four decode steps, hits and misses.
        dict(name="slots_qwen3_q8", kind="slots", dtype="q8", experts=64, slots=24, steps=4, top_k=8,
             d_model=2048, d_ff=768, zipf=1.0),
        # Prefill of a short prompt (64 tokens), skewed expert popularity.
        dict(name="prefill_qwen3_q8_64", kind="prefill", dtype="q8", qmm=False, experts=128, top_k=8, tokens=64,
             d_model=2048, d_ff=768, zipf=1.1),
        # Prefill chunk in the engine's default Q4_0 arithmetic, with a
        # prompt length that fits no tile.
        dict(name="prefill_mixtral_q4_qmm_333", kind="prefill", dtype="q4", qmm=True, experts=8, top_k=2, tokens=333,
             d_model=4096, d_ff=14336, zipf=0.0),
        # The largest chunk the grouped call takes (4096 routed pairs): few
        # large experts, ...
        dict(name="prefill_mixtral_q4_2048", kind="prefill", dtype="q4", qmm=False, experts=8, top_k=2, tokens=2048,
             d_model=4096, d_ff=14336, zipf=0.0),
        # ... and many, with a residual stream's worth of tokens per expert
        # that varies widely.
        dict(name="prefill_deepseek_q4_512", kind="prefill", dtype="q4", qmm=False, experts=256, top_k=8, tokens=512,
             d_model=7168, d_ff=2048, zipf=1.0),
        # Routing of a prefill chunk on the GPU.
        dict(name="router_qwen3_2048", kind="router", experts=128, top_k=8, tokens=2048, d_model=2048, sigmoid=False,
             groups=1),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["stack", "layer", "expert", "views", "slots", "prefill", "prefill", "prefill", "router"])
    dtype = rng.choice(["q4", "q8"])
    dm, dff = 64 * _logint(rng, 8, 112), 64 * _logint(rng, 6, 224)
    zipf = rng.choice([0.0, rng.uniform(0.5, 1.2)])
    if kind == "router":
        experts = rng.choice([8, 60, 64, 128, 160, 256])
        groups = rng.choice([1, 4]) if experts >= 60 else 1
        return dict(kind=kind, experts=experts, top_k=rng.randint(1, 8), tokens=_logint(rng, 1, 4096),
                    d_model=rng.choice([dm, dm + rng.randint(1, 31)]), sigmoid=rng.random() < 0.4, groups=groups)
    qmm = dtype == "q4" and rng.random() < 0.4
    if kind == "expert":
        return dict(kind=kind, dtype=dtype, qmm=qmm, d_model=dm, d_ff=dff)
    experts = _logint(rng, 8, 128)
    expert_bytes = 3 * dm * dff // 32 * BLOCK_BYTES[dtype]
    while experts > 8 and experts * expert_bytes > 6 << 30:
        experts //= 2
    experts = max(experts, 8)
    if kind == "views":
        return dict(kind=kind, dtype=dtype, experts=experts, n=rng.randint(1, 8), d_model=dm, d_ff=dff)
    top_k = rng.randint(1, 8)
    if kind == "slots":
        return dict(kind=kind, dtype="q8", experts=64, slots=rng.randint(17, 40), steps=rng.randint(2, 4), top_k=top_k,
                    d_model=64 * rng.randint(8, 32), d_ff=64 * rng.randint(6, 12), zipf=zipf)
    if kind == "stack":
        layers = _logint(rng, 2, 32)
        while layers > 1 and layers * experts * expert_bytes > 12 << 30:
            layers //= 2
        return dict(kind=kind, dtype=dtype, layers=layers, experts=experts, top_k=top_k, tokens=1, d_model=dm,
                    d_ff=dff, zipf=zipf)
    if kind == "layer":
        return dict(kind=kind, dtype=dtype, qmm=qmm, experts=experts, top_k=top_k, tokens=_logint(rng, 1, 8),
                    d_model=dm, d_ff=dff, zipf=zipf)
    tokens = _logint(rng, 2, 2048)
    while tokens > 1 and (tokens * top_k > 4096 or tokens * top_k * dm * dff > 4096 * 4096 * 14336):
        tokens = tokens * 2 // 3
    return dict(kind=kind, dtype=dtype, qmm=qmm, experts=experts, top_k=top_k, tokens=tokens, d_model=dm, d_ff=dff,
                zipf=zipf)


# ---- inputs --------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _blobs(g, dtype, n, d_model, d_ff):
    """n expert blobs, [n, expert bytes] uint8."""
    bb = BLOCK_BYTES[dtype]
    blocks = n * 3 * d_model * d_ff // 32
    b = torch.empty(blocks, bb, dtype=torch.uint8, device=DEV).random_(0, 256, generator=g)
    if dtype == "q8":
        b.view(torch.int8).clamp_(min=-127)
    lo, hi = (0.005, 0.02) if dtype == "q4" else (0.002, 0.01)
    d = torch.empty(blocks, 1, device=DEV).uniform_(lo, hi, generator=g)
    b[:, :2] = d.to(torch.float16).view(torch.uint8)
    return b.view(n, -1)


def _table(blobs):
    step = blobs.shape[1]
    return blobs.data_ptr() + step * torch.arange(blobs.shape[0], dtype=torch.int64, device=DEV)


def _routes(g, tokens, experts, top_k, zipf):
    popularity = -zipf * torch.log(torch.arange(1, experts + 1, device=DEV, dtype=torch.float32))
    logits = torch.randn(tokens, experts, generator=g, device=DEV)
    logits += popularity[torch.randperm(experts, generator=g, device=DEV)]
    v, ids = logits.topk(top_k, dim=1)
    return ids.to(torch.int32).contiguous(), torch.softmax(v, 1).contiguous()


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    dm = case["d_model"]
    s = dict(case=case)
    if kind == "router":
        s["gate"] = 0.02 * torch.randn(case["experts"], dm, generator=g, device=DEV)
        s["x"] = torch.randn(case["tokens"], dm, generator=g, device=DEV)
        s["bias"] = 0.01 * torch.randn(case["experts"], generator=g, device=DEV) if case["sigmoid"] else None
        return s
    dff, dtype = case["d_ff"], case["dtype"]
    if kind == "expert":
        s["blob"] = _blobs(g, dtype, 1, dm, dff)[0]
        s["x"] = torch.randn(dm, generator=g, device=DEV)
        return s
    n = case["experts"]
    if kind == "slots":
        dev = _blobs(g, dtype, n, dm, dff)
        host = torch.empty(dev.shape, dtype=torch.uint8, pin_memory=True)
        host.copy_(dev)
        s["host"] = [host[e] for e in range(n)]
        s["cache"] = mer.SlotCache(DTYPES[dtype], dm, dff, case["slots"], n)
        s["steps"] = []
        for _ in range(case["steps"]):
            ids, w = _routes(g, 1, n, case["top_k"], case["zipf"])
            s["steps"].append((ids, ids[0].tolist(), w, torch.randn(1, dm, generator=g, device=DEV)))
        return s
    layers = case.get("layers", 1)
    s["blobs"] = _blobs(g, dtype, layers * n, dm, dff)
    table = _table(s["blobs"])
    if kind == "views":
        s["table"] = table
        s["ids"] = torch.randperm(n, generator=g, device=DEV)[:case["n"]].to(torch.int32)
        s["x"] = torch.randn(dm, generator=g, device=DEV).to(torch.float16)
        return s
    s["layers"] = []
    for l in range(layers):
        ids, w = _routes(g, case["tokens"], n, case["top_k"], case["zipf"])
        x = torch.randn(case["tokens"], dm, generator=g, device=DEV)
        s["layers"].append(dict(table=table[l * n:(l + 1) * n].clone(), ids=ids, weights=w, x=x,
                                out=torch.empty_like(x)))
    return s


# ---- one pass ------------------------------------------------------------

def run(state):
    c = state["case"]
    kind, dm = c["kind"], c["d_model"]
    if kind == "router":
        return routing.route_linear_gate_gpu(state["gate"], state["x"], c["top_k"], sigmoid=c["sigmoid"],
                                             bias=state["bias"], n_group=c["groups"],
                                             topk_group=max(1, c["groups"] // 2), return_logits=True)
    dtype, dff = DTYPES[c["dtype"]], c["d_ff"]
    if kind == "expert":
        return mer.dispatch_expert_forward(dtype, state["blob"], state["x"], dm, dff, use_qmm=c["qmm"])
    if kind == "views":
        return mer.routed_expert_matmul_batch(dtype, dm, dff, state["table"], state["ids"], state["x"])
    if kind == "slots":
        outs = []
        for ids, host_ids, w, x in state["steps"]:
            state["cache"].prepare(host_ids, host_blobs=[state["host"][e] for e in host_ids])
            outs.append(mer.moe_forward(dtype, dm, dff, state["cache"], ids, w, x))
        return outs
    if kind == "stack":
        mer.moe_forward_layers(dtype, dm, dff, state["layers"])
        return [la["out"] for la in state["layers"]]
    la = state["layers"][0]
    fn = mer.moe_grouped if kind == "prefill" else mer.moe_forward
    return fn(dtype, dm, dff, la["table"], la["ids"], la["weights"], la["x"], qmm=c["qmm"])


# ---- what a pass cannot do without ---------------------------------------

def _distinct(tokens, experts, top_k, zipf):
    """Expected distinct experts of a layer, by their share of the draws."""
    p = [r ** -zipf for r in range(1, experts + 1)]
    total = sum(p)
    return min(experts, max(top_k, sum(1.0 - (1.0 - min(1.0, top_k * q / total)) ** tokens for q in p)))


def work(case):
    kind, dm = case["kind"], case["d_model"]
    if kind == "router":
        t, e = case["tokens"], case["experts"]
        return {"bytes": 4 * (e * dm + t * dm + t * e + 2 * t * case["top_k"]), "flops": 2 * t * e * dm}
    dff = case["d_ff"]
    expert = 3 * dm * dff // 32 * BLOCK_BYTES[case["dtype"]]
    pair = 6 * dm * dff
    if kind == "expert":
        return {"bytes": expert + 8 * dm, "flops": pair}
    if kind == "views":
        n = case["n"]
        return {"bytes": n * expert + 2 * dm * (n + 1), "flops": n * pair}
    k = case["top_k"]
    if kind == "slots":
        return {"bytes": case["steps"] * (k * expert + 8 * dm), "flops": case["steps"] * k * pair}
    t, layers = case["tokens"], case.get("layers", 1)
    u = _distinct(t, case["experts"], k, case["zipf"])
    return {"bytes": int(layers * (u * expert + 8 * t * dm)), "flops": layers * t * k * pair}


def tolerance(case):
    if case["kind"] == "router":
        # f32 dot products in another order; a near tie may pick the other expert
        return {"rel": 1e-6, "differ": 5e-4}
    if case["kind"] == "views":
        return {"rel": 8e-4}  # f16 outputs
    if case.get("qmm"):
        # the inner activation is rounded to 8 bits: an element near a
        # midpoint may round either way, one step of one element each
        return {"rel": 2e-3}
    return {"rel": 2e-6}


# ---- the same in 64 bits -------------------------------------------------

def _dequant(blob, dtype, d_model, d_ff):
    """(gate [d_ff, d_model], up, down [d_model, d_ff]) in float64."""
    b = blob.view(3, -1, BLOCK_BYTES[dtype])
    d = b[:, :, :2].contiguous().view(torch.float16).to(torch.float64)
    if dtype == "q4":
        q = torch.cat([b[:, :, 2:] & 15, b[:, :, 2:] >> 4], 2).to(torch.float64) - 8
    else:
        q = b[:, :, 2:].contiguous().view(torch.int8).to(torch.float64)
    w = (d * q).view(3, -1)
    return w[0].view(d_ff, d_model), w[1].view(d_ff, d_model), w[2].view(d_model, d_ff)


def _q8_activation(v):
    """Q8_0 rounding of an activation, per 32 values: d = max / 127 kept as
    f16, q rounded half away from zero."""
    b = v.to(torch.float32).view(v.shape[0], -1, 32)
    d = b.abs().amax(2, keepdim=True) / 127.0
    inv = torch.where(d != 0, 1.0 / d, torch.zeros_like(d))
    t = b * inv
    q = torch.sign(t) * torch.floor(t.abs().to(torch.float64) + 0.5)
    return (q * d.to(torch.float16).to(torch.float64)).view(v.shape)


def _ffn(blob, dtype, d_model, d_ff, x, qmm=False):
    """x [n, d_model] float64 -> y [n, d_model] float64."""
    gate, up, down = _dequant(blob, dtype, d_model, d_ff)
    if qmm:
        x = _q8_activation(x)
    a, u = x @ gate.t(), x @ up.t()
    h = a * torch.sigmoid(a) * u
    if qmm:
        h = _q8_activation(h)
    return h @ down.t()


def _moe(expert, dtype, d_model, d_ff, ids, w, x, qmm=False):
    x64 = x.to(torch.float64)
    out = torch.zeros_like(x64)
    for e in ids.unique().tolist():
        t, k = (ids == e).nonzero(as_tuple=True)
        y = _ffn(expert(e), dtype, d_model, d_ff, x64[t], qmm)
        out.index_add_(0, t, y * w[t, k].to(torch.float64)[:, None])
    return out


def exact(case, seed):
    s = prepare(case, seed)
    kind, dm = case["kind"], case["d_model"]
    if kind == "router":
        logits = s["x"].to(torch.float64) @ s["gate"].to(torch.float64).t()
        score = torch.sigmoid(logits) if case["sigmoid"] else torch.softmax(logits, 1)
        sel = score if s["bias"] is None else score + s["bias"].to(torch.float64)
        if case["groups"] > 1:
            per = sel.view(sel.shape[0], case["groups"], -1)
            best = per.topk(2, dim=2).values.sum(2).topk(max(1, case["groups"] // 2), dim=1).indices
            keep = torch.zeros(per.shape[:2], dtype=torch.bool, device=DEV).scatter_(1, best, True)
            sel = torch.where(keep[:, :, None], per, torch.full_like(per, -math.inf)).view(sel.shape)
        ids = sel.topk(case["top_k"], dim=1).indices
        w = score.gather(1, ids)
        return ids.to(torch.int32), w / w.sum(1, keepdim=True), logits
    dff, dtype = case["d_ff"], case["dtype"]
    if kind == "expert":
        return _ffn(s["blob"], dtype, dm, dff, s["x"][None].to(torch.float64), case["qmm"])[0]
    if kind == "views":
        x = s["x"][None].to(torch.float64)
        return torch.cat([_ffn(s["blobs"][e], dtype, dm, dff, x) for e in s["ids"].tolist()])
    if kind == "slots":
        return [_moe(lambda e: s["host"][e].to(DEV), dtype, dm, dff, ids, w, x) for ids, _, w, x in s["steps"]]
    n = case["experts"]
    outs = [_moe(lambda e, l=l: s["blobs"][l * n + e], dtype, dm, dff, la["ids"], la["weights"], la["x"],
                 case.get("qmm", False)) for l, la in enumerate(s["layers"])]
    return outs if kind == "stack" else outs[0]
