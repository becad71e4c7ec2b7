"""The calls that programs on this framework make, as measurable cases.

Three programs stand behind them: a decoder that serves a batch of sequences one token at a
time, a server that mixes prompt chunks with decoding sequences in one packed batch, and a
prefill of whole prompts. Each calls the MoE layer (router, dispatch, grouped SwiGLU FFN,
combine with the skip residual), the dispatch operator on a routing of its own, the YvMoEGate
router, or the two norms in front of the layer. Layer shapes are those of the benchmark's
configurations; drawn cases add hidden and FFN widths that are any multiple of the block the
weight format allows, and token counts over the whole range from one to a long prefill.

``listed`` gives the fixed cases, ``draw`` more of the same ranges, ``prepare`` what a program
has in hand before the call, ``run`` one call, ``work`` the bytes and operations it cannot do
without, ``exact`` its result in 64 bits by plain torch, ``tolerance`` how far another correct
implementation may be from it.
"""
import math

import torch

from pisceslx_amd import _lib
from pisceslx_amd import functional as yvf
from pisceslx_amd.dispatch import PiscesLxFusedMoEDispatch
from pisceslx_amd.gate import YvMoEGate, YvStableMoEGate
from pisceslx_amd.norms import YvRMSNorm, rms_norm_chain
from pisceslx_amd.quant import ExpertPacker, FORMAT_BY_NAME

# hidden, experts, ffn, top_k, shared experts of the benchmark's layers, and the most tokens a
# drawn call of each takes
SHAPES = {
    "small": (1024, 8, 2816, 2, 1, 4096),
    "mid": (4096, 64, 1408, 6, 2, 16721),
    "wide": (5120, 128, 1536, 8, 1, 8192),
    "huge": (7168, 256, 2048, 8, 0, 8192),
}


def _layer(name, op, shape, fmt, tokens, fixed=False, **sizes):
    H, E, Fd, k, S, _ = SHAPES[shape]
    c = {"name": name, "op": op, "hidden": H, "experts": E, "ffn": Fd, "top_k": k, "shared": S,
         "format": fmt, "tokens": tokens, "fixed": fixed}
    c.update(sizes)
    return c


def listed():
    return [
        # one decode step of 64 sequences: the two norms in front of the MoE layer
        {"name": "norms_decode", "op": "norms", "hidden": 4096, "tokens": 64, "format": "bf16"},
        # the same over a packed prefill of 32 prompts
        {"name": "norms_prefill", "op": "norms", "hidden": 4096, "tokens": 16721, "format": "bf16"},
        # the router the reference's layers build, one decode step and one long prompt
        {"name": "moegate_decode", "op": "moegate", "hidden": 4096, "experts": 64, "top_k": 6,
         "tokens": 64, "batch": 64, "format": "bf16"},
        {"name": "moegate_prefill", "op": "moegate", "hidden": 4096, "experts": 64, "top_k": 6,
         "tokens": 16721, "batch": 1, "format": "bf16"},
        # one user, one token
        _layer("layer_int8_1", "layer", "mid", "int8", 1),
        # a decode step of 64 sequences
        _layer("layer_int8_64", "layer", "mid", "int8", 64),
        # a server's mixed batch: a prompt chunk of 512 with 188 decoding sequences
        _layer("layer_int8_700", "layer", "mid", "int8", 700),
        # packed prefill of 32 prompts of log-normal lengths
        _layer("layer_int8_16721", "layer", "mid", "int8", 16721),
        # eight prompt chunks of 512 with 248 decoding sequences on int4 weights
        _layer("layer_int4_4344", "layer", "wide", "int4", 4344),
        # fixed-shape routing with a skewed expert bias on fp8 weights
        _layer("layer_fp8_8192", "layer", "huge", "fp8", 8192, fixed=True),
        # the unquantized fp32 layer on 16 ragged prompts
        _layer("layer_f32_2052", "layer", "small", "f32", 2052),
        # the dispatch operator on unquantized bf16 experts, the default of a bf16 layer, for a
        # mid-sized decode batch routed by the caller
        _layer("dispatch_bf16_333", "dispatch", "mid", "bf16", 333, shared=0),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(["norms", "moegate", "layer", "layer", "layer", "layer", "dispatch", "dispatch"])
    if op == "norms":
        return {"op": op, "hidden": 64 * _log_int(rng, 8, 128), "tokens": _log_int(rng, 1, 16721),
                "format": rng.choice(["bf16", "bf16", "f32"])}
    if op == "moegate":
        n = _log_int(rng, 1, 16721)
        return {"op": op, "hidden": rng.choice([1024, 2048, 4096]), "experts": rng.choice([8, 48, 64, 128]),
                "top_k": rng.choice([2, 6, 8]), "tokens": n, "batch": n if rng.random() < 0.5 else 1,
                "format": "bf16"}
    shape = rng.choice(["small", "mid", "mid", "wide", "huge"])
    H, E, Fd, k, S, most = SHAPES[shape]
    fmts = {"small": ["f32", "f32", "bf16", "int8"], "mid": ["int8", "int8", "int4", "fp8", "bf16"],
            "wide": ["int4", "int4", "int8", "bf16"], "huge": ["fp8"]}[shape]
    fmt = rng.choice(fmts)
    c = _layer("", op, shape, fmt, _log_int(rng, 1, most), fixed=shape == "huge" or rng.random() < 0.25)
    del c["name"]
    if op == "dispatch":
        c["shared"] = 0
    if shape != "huge" and rng.random() < 0.3:  # widths of no configuration
        step = 128 if fmt in ("int4", "fp8") else 64
        c["hidden"] = step * rng.randint(640 // step, H // step)
        c["ffn"] = step * rng.randint(512 // step, Fd // step)
    return c


def _dtype(c):
    return torch.float32 if c["format"] == "f32" else torch.bfloat16


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


# ---------------------------------------------------------------- inputs, the same for run and exact
def _norm_inputs(c, seed):
    g, dt = _gen(seed), _dtype(c)
    x = (_randn(g, c["tokens"], c["hidden"]) * 1.5).to(dt)
    w1 = (1.0 + 0.1 * _randn(g, c["hidden"])).to(dt)
    w2 = (1.0 + 0.1 * _randn(g, c["hidden"])).to(dt)
    return x, w1, w2


def _moegate_inputs(c, seed):
    """Activations after a norm, and the gate's parameters by name (scaled as initialised)."""
    g, dt = _gen(seed), _dtype(c)
    H, E = c["hidden"], c["experts"]
    D = max(64, H // 64)
    x = _randn(g, c["tokens"], H).to(dt)
    lin = lambda o, i: ((torch.rand(o, i, generator=g, device="cuda") * 2 - 1) / math.sqrt(i)).to(dt)
    p = {"gate.weight": lin(E, H), "hicl_dg_encoder.dg_proj.weight": lin(4 * H, H),
         "hicl_prototypes": (_randn(g, E, 4 * H) * 0.02).to(dt), "got_cluster_proj.weight": lin(E, H),
         "gate_k.weight": lin(E, H), "gate_v.weight": lin(E, H),
         "expert_embeddings": _randn(g, E, D).to(dt),
         "input_encoder.0.weight": lin(D, H), "input_encoder.2.weight": lin(D, D),
         "expert_capability_encoder.0.weight": lin(D, D), "expert_capability_encoder.2.weight": lin(D, D),
         "expert_bias": (_randn(g, E) * 0.05).to(dt)}
    return x, p


def _router_inputs(c, seed):
    g, dt = _gen(seed), _dtype(c)
    N, H, E = c["tokens"], c["hidden"], c["experts"]
    r = {"x": _randn(g, N, H).to(dt), "skip": (_randn(g, N, H) * 0.1).to(dt),
         "gate": (_randn(g, E, H) * 0.02).to(dt)}
    if c["op"] == "dispatch":  # the caller's routing: distinct experts per token, weights that sum to 1
        logits = _randn(g, N, E) * 1.3
        top = torch.topk(logits, c["top_k"], dim=1)
        r["indices"] = top.indices.contiguous()
        r["weights"] = torch.softmax(top.values, dim=1).contiguous()
    if c["fixed"]:  # a skewed expert bias: Zipf shares over a shuffled order
        order = torch.randperm(E, generator=g, device="cuda")
        r["bias"] = torch.empty(E, device="cuda")
        r["bias"][order] = -1.2 * torch.log(torch.arange(1, E + 1, device="cuda").float())
    else:
        r["w1"], r["w2"] = _randn(g, 64, H) * 0.02, _randn(g, 1, 64) * 0.02
    return r


def _expert_weights(c, seed):
    """(gate, up, down) of one expert after the other, routed first, then shared."""
    g = _gen(seed + 7919)
    H, Fd = c["hidden"], c["ffn"]
    for _ in range(c["experts"] + c["shared"]):
        yield tuple(_randn(g, o, i) * 0.02 for o, i in ((Fd, H), (Fd, H), (H, Fd)))


def _mix(c):
    S = c["shared"]
    return torch.full((S,), 1.0 / S, device="cuda") if S else None


# ---------------------------------------------------------------- what a program has in hand
@torch.no_grad()
def prepare(case, seed):
    c = case
    dt = _dtype(c)
    act = _lib.ACT_F32 if dt == torch.float32 else _lib.ACT_BF16
    if c["op"] == "norms":
        x, w1, w2 = _norm_inputs(c, seed)
        norms = []
        for w in (w1, w2):
            n = YvRMSNorm(c["hidden"], device="cuda", dtype=dt).eval()
            n.weight.copy_(w)
            norms.append(n)
        return {"case": c, "x": x, "norms": norms}
    if c["op"] == "moegate":
        x, p = _moegate_inputs(c, seed)
        cfg = type("Cfg", (), {"path_moe_stage_size": 1})()
        gate = YvMoEGate(c["hidden"], c["experts"], top_k=c["top_k"], device="cuda", dtype=dt, cfg=cfg).eval()
        gate.load_state_dict(p, strict=False)
        return {"case": c, "x": x.view(c["batch"], -1, c["hidden"]), "gate": gate}
    r = _router_inputs(c, seed)
    pk = ExpertPacker(FORMAT_BY_NAME[c["format"]], c["experts"], c["shared"], c["hidden"], c["ffn"], "cuda")
    for i, ws in enumerate(_expert_weights(c, seed)):
        pk.set(i, *ws)
    if c["op"] == "dispatch":
        op = PiscesLxFusedMoEDispatch(c["experts"], c["top_k"]).eval()
        op.check_indices = False
        return {"case": c, "x": r["x"], "weights": r["weights"], "indices": r["indices"], "op": op,
                "experts": pk.packed}
    gate = YvStableMoEGate(c["hidden"], c["experts"], top_k=c["top_k"], device="cuda", dtype=dt,
                           fixed_shape_mode=c["fixed"], enable_dynamic_capacity=not c["fixed"]).eval()
    gate.gate.weight.copy_(r["gate"])
    if c["fixed"]:
        gate.expert_bias.copy_(r["bias"])
    else:
        gate.complexity_predictor[0].weight.copy_(r["w1"])
        gate.complexity_predictor[0].bias.zero_()
        gate.complexity_predictor[2].weight.copy_(r["w2"])
        gate.complexity_predictor[2].bias.zero_()
    st = gate.router_state(act)
    ws = torch.empty(max(256, yvf.workspace_bytes(c["tokens"], act, st, pk.packed)), dtype=torch.uint8,
                     device="cuda")
    return {"case": c, "x": r["x"], "skip": r["skip"] if c["shared"] else None, "gate": gate, "act": act,
            "experts": pk.packed, "mix": _mix(c), "workspace": ws}


@torch.no_grad()
def run(state):
    op = state["case"]["op"]
    if op == "norms":
        return rms_norm_chain(state["x"], *state["norms"])
    if op == "moegate":
        weights, indices, loss = state["gate"](state["x"])
        return {"weights": weights, "indices": indices, "loss": loss, "logits": state["gate"].last_logits}
    if op == "dispatch":
        return state["op"](state["x"], state["weights"], state["indices"], state["experts"])
    out, shared, routing = yvf.moe_forward(state["x"], state["gate"].router_state(state["act"]),
                                           state["experts"], state["mix"], state["skip"],
                                           workspace=state["workspace"])
    res = {"out": out, "weights": routing.weights, "indices": routing.indices}
    if shared is not None:
        res["shared"] = shared
    return res


# ---------------------------------------------------------------- bytes and operations
def _expert_shares(c):
    """Each expert's chance to be among a token's top k: its bias plus a normal logit (of the
    standard deviation that the inputs give) above the level that k experts reach on average."""
    E, k = c["experts"], c["top_k"]
    if not c["fixed"] or c["op"] == "dispatch" or k == E:
        return [k / E] * E
    sd = 0.02 * math.sqrt(c["hidden"])
    bias = [-1.2 * math.log(i + 1) for i in range(E)]
    shares = lambda level: [0.5 * math.erfc((level - b) / (sd * math.sqrt(2.0))) for b in bias]
    lo, hi = -40.0, 40.0
    for _ in range(60):
        mid = 0.5 * (lo + hi)
        lo, hi = (mid, hi) if sum(shares(mid)) > k else (lo, mid)
    return shares(lo)


def work(case):
    c = case
    N, H = c["tokens"], c["hidden"]
    b = 4 if c["format"] == "f32" else 2
    if c["op"] == "norms":
        return {"bytes": 2 * N * H * b + 2 * H * b, "flops": 8 * N * H}
    E, k = c["experts"], c["top_k"]
    if c["op"] == "moegate":
        rows = 4 * H + 4 * E + max(64, H // 64)
        return {"bytes": rows * H * b + E * 4 * H * b + N * H * b + N * E * 4 + N * k * (b + 8),
                "flops": 2 * N * H * rows}
    Fd, S = c["ffn"], c["shared"]
    active = sum(1.0 - (1.0 - q) ** N for q in _expert_shares(c))  # experts that receive a token
    per = 3 * H * Fd
    expert = {"f32": 4 * per, "bf16": 2 * per, "int8": per + 2 * (2 * Fd + H),
              "int4": per // 2 + 2 * (per // 128), "fp8": per + 4 * (per // 16384)}[c["format"]]
    nbytes = (active + S) * expert + 2 * N * H * b
    flops = 6 * H * Fd * N * (k + S)
    if c["op"] == "dispatch":
        return {"bytes": int(nbytes) + N * k * 12, "flops": flops}
    nbytes += E * H * b + N * k * 12 + (2 * N * H * b if S else 0)  # + shared output and skip
    flops += 2 * N * H * E
    if not c["fixed"]:
        nbytes += 64 * H * 4
        flops += 2 * N * H * 64
    return {"bytes": int(nbytes), "flops": flops}


def tolerance(case):
    if case["op"] == "norms":
        return {"rel": 1e-2 if case["format"] == "bf16" else 5e-7}
    if case["op"] == "moegate":
        # weights are rounded to bf16, logits are fp32; near-ties may pick another expert
        return {"rel": 8e-3, "differ": 1e-3}
    if case["format"] == "f32":
        return {"rel": 5e-6, "differ": 1e-3}
    # bf16 activations, h and outputs are rounded to bf16
    return {"rel": 1.5e-2, "differ": 1e-3}


# ---------------------------------------------------------------- 64-bit results in plain torch
def _stored(w, fmt):
    """The values the format stores for w, in 64 bits."""
    if fmt == "f32":
        return w.double()
    if fmt == "bf16":
        return w.to(torch.bfloat16).double()
    o, i = w.shape
    if fmt == "int8":
        s = (w.abs().amax(dim=1) / 127.0).clamp(min=1e-8).to(torch.bfloat16)
        return torch.round(w / s.float()[:, None]).clamp(-128, 127).double() * s.double()[:, None]
    if fmt == "int4":
        v = w.view(o, i // 128, 128)
        s = (v.abs().amax(dim=-1) / 7.0).clamp(min=1e-8).to(torch.bfloat16)
        q = (torch.round(v / s.float()[..., None]) + 8).clamp(0, 15).double() - 8.0
        return (q * s.double()[..., None]).view(o, i)
    v = w.view(o // 128, 128, i // 128, 128)
    s = (v.abs().amax(dim=(1, 3)) / 448.0).clamp(min=1e-12)[:, None, :, None]
    q = (v / s).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
    return (q.double() * s.double()).view(o, i)


def _exact_norms(c, seed):
    x, w1, w2 = (t.double() for t in _norm_inputs(c, seed))
    for w in (w1, w2):
        x = x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + 1e-6) * w
    return x


def _exact_moegate(c, seed):
    x, p = _moegate_inputs(c, seed)
    p = {n: t.double() for n, t in p.items()}
    bf = lambda v: float(torch.tensor(v, dtype=torch.bfloat16))  # scalar parameters are bf16 tensors
    silu = torch.nn.functional.silu
    logits = []
    soft_total = 0.0
    eff = torch.tensor(3.0, dtype=torch.bfloat16)
    if c["tokens"] // c["batch"] >= 8192:
        eff = eff * 0.3
    eff = float(eff)
    ee = silu(p["expert_embeddings"] @ p["expert_capability_encoder.0.weight"].t()) \
        @ p["expert_capability_encoder.2.weight"].t()
    for xs in x.split(4096):
        xs = xs.double()
        dg = torch.relu(xs @ p["hicl_dg_encoder.dg_proj.weight"].t())
        top = torch.topk(dg, 32, dim=1)
        sparse = torch.zeros_like(dg).scatter_(1, top.indices, top.values)
        sparse = sparse / sparse.norm(dim=1, keepdim=True).clamp(min=1e-12)
        lk, lv = xs @ p["gate_k.weight"].t(), xs @ p["gate_v.weight"].t()
        soft = torch.sigmoid(lk - lk.median(dim=1, keepdim=True).values) * torch.softmax(lv, dim=1)
        soft = soft / soft.sum(dim=1, keepdim=True).clamp(min=10 * 2.0 ** -7)
        soft_total += float(soft.sum())
        ie = silu(xs @ p["input_encoder.0.weight"].t()) @ p["input_encoder.2.weight"].t()
        z = xs @ p["gate.weight"].t() + bf(0.1) * (sparse @ p["hicl_prototypes"].t()) \
            + bf(0.05) * (xs @ p["got_cluster_proj.weight"].t() + soft + ie @ ee.t()) + p["expert_bias"]
        logits.append(z / eff)
    z = torch.cat(logits)
    scores = torch.softmax(z, dim=1)
    top = torch.topk(scores, c["top_k"], dim=1)
    budget = bf(float(c["top_k"]))
    loss = 0.01 * ((scores.mean(dim=0) - 1.0 / c["experts"]) ** 2).sum() + 1e-4 * (z * z).mean() \
        + 0.01 * (soft_total / c["tokens"] - budget) ** 2
    return {"weights": torch.softmax(top.values, dim=1), "indices": top.indices, "loss": loss, "logits": z}


def _exact_routing(c, r):
    """YvStableMoEGate in 64 bits: softmax, top-k, softmax of the k, then the capacity trim."""
    x, E, N, k = r["x"].double(), c["experts"], c["tokens"], c["top_k"]
    z = x @ r["gate"].double().t()
    if c["fixed"]:
        z = z + r["bias"].double()
    p = torch.softmax(z, dim=1)
    top = torch.topk(p, k, dim=1)
    w = torch.softmax(top.values, dim=1)
    if c["fixed"]:
        return w, top.indices
    score = torch.sigmoid(torch.relu(x @ r["w1"].double().t()) @ r["w2"].double().t()).mean()
    factor = min(2.0, max(0.5, 0.5 + 1.5 * float(score)))
    cap = max(int(N * factor / E), 4)
    # rank of each slot among its expert's, by probability (ties by token): the first cap stay
    flat = top.indices.reshape(-1)
    by_p = torch.argsort(top.values.reshape(-1), descending=True, stable=True)
    order = by_p[torch.argsort(flat[by_p], stable=True)]
    counts = torch.bincount(flat, minlength=E)
    first = torch.cumsum(counts, 0) - counts
    rank = torch.empty_like(flat)
    rank[order] = torch.arange(flat.numel(), device=flat.device) - first[flat[order]]
    w = w * (rank < cap).view(N, k)
    return w / w.sum(dim=1, keepdim=True).clamp(min=1e-8), top.indices


def _exact_ffn(c, seed, x, w, idx):
    """Weighted sum of the routed experts' outputs, and the shared experts' mixture."""
    out, shared = torch.zeros_like(x), torch.zeros_like(x)
    for e, ws in enumerate(_expert_weights(c, seed)):
        if e < c["experts"]:
            t, slot = torch.nonzero(idx == e, as_tuple=True)
            if t.numel() == 0:
                continue
        g, u, d = (_stored(m, c["format"]) for m in ws)
        xs = x[t] if e < c["experts"] else x
        y = (torch.nn.functional.silu(xs @ g.t()) * (xs @ u.t())) @ d.t()
        if e < c["experts"]:
            out.index_add_(0, t, w[t, slot, None] * y)
        else:
            shared += y / c["shared"]
    return out, shared


@torch.no_grad()
def exact(case, seed):
    c = case
    if c["op"] == "norms":
        return _exact_norms(c, seed)
    if c["op"] == "moegate":
        return _exact_moegate(c, seed)
    r = _router_inputs(c, seed)
    x = r["x"].double()
    if c["op"] == "dispatch":
        return _exact_ffn(c, seed, x, r["weights"].double(), r["indices"])[0]
    w, idx = _exact_routing(c, r)
    out, shared = _exact_ffn(c, seed, x, w, idx)
    res = {"out": out, "weights": w, "indices": idx}
    if c["shared"]:
        res["out"] = out + shared + 0.1 * r["skip"].double()
        res["shared"] = shared
    return res
