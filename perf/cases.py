"""Performance cases of the U4 MoE expert path, through the public entry points.

A case is a dict of plain values; its "kind" names the work:

* ``fc``           the U4 fixed FC of one token: 1 to 4 matrices over one input
* ``lm_head``      the U4 LM head of one token with its top-k
* ``decode_block`` one decode FFN block as a per-layer loop calls it between two
                   attention blocks: RMSNorm, device router, MoE FFN + residual
* ``decode_plan``  one token through a resident layer stack, routes from logits
* ``routed_plan``  the same with every layer routed from its own input
* ``routed_stack`` the same without a plan (any layer shape)
* ``prefill``      the MoE FFN block of a batch of tokens, given routes
* ``run_layer``    the routed sum alone: f32 activations, strided top-k ids
* ``fused_op``     router logits in, block output and routes out, separate gate
                   and up projections
* ``router``       the f32 router of a batch of tokens with its selection
* ``prefill_stack`` a batch of tokens through several layers

Weights, activations and routings follow the distributions of
``aima_u4moe.synth``; everything is made on the GPU from the seed alone.
"""

import math

import torch

import __graft_entry__

pkg = __graft_entry__.load_package()
synth = pkg.synth

EPS = 1e-6
MIN_SUM = pkg.MIN_WEIGHT_SUM
DEV = "cuda"


def listed():
    return [
        # the smallest call: shared-expert gate scalar, shared gate, shared up
        # and router over one token, four projections of one input
        {"name": "fc fanout", "kind": "fc", "k": 2048, "rows": "1,512,512,256", "group": 128},
        # a whole vocabulary for one token: the largest single matrix
        {"name": "lm head top-8", "kind": "lm_head", "k": 2048, "rows": 248320, "group": 128,
         "topk": 8},
        # one layer of batch-1 decode in an engine that runs attention between
        {"name": "decode block", "kind": "decode_block", "hidden": 2048, "inter": 512,
         "experts": 256, "group": 128, "topk": 8},
        # the benchmark's headline: a token through all 40 layers
        {"name": "decode plan 40 layers", "kind": "decode_plan", "layers": 40, "hidden": 2048,
         "inter": 512, "experts": 256, "group": 128, "topk": 8},
        # true decode, where the routes depend on the layer before
        {"name": "routed plan 4 layers", "kind": "routed_plan", "layers": 4, "hidden": 2048,
         "inter": 512, "experts": 256, "group": 128, "topk": 8},
        # true decode of a shape that the resident plan does not take
        {"name": "routed stack 4 layers", "kind": "routed_stack", "layers": 4, "hidden": 1024,
         "inter": 256, "experts": 64, "group": 64, "topk": 4},
        # a few tokens at once: a short prompt's tail, a batch of decode
        # streams, a draft being checked
        {"name": "prefill T=7", "kind": "prefill", "tokens": 7, "hidden": 2048, "inter": 512,
         "experts": 256, "topk": 8, "zipf": 0.0, "residual": True},
        # a short prompt: every expert has a few rows
        {"name": "fused op T=96", "kind": "fused_op", "tokens": 96, "hidden": 2048, "inter": 512,
         "experts": 256, "topk": 8, "shared": True},
        # an ordinary ragged prompt through the routed-only layer
        {"name": "run layer T=777", "kind": "run_layer", "tokens": 777, "hidden": 2048,
         "inter": 512, "experts": 256, "topk": 8, "pad": 2},
        # the benchmark's prefill chunk, experts of skewed popularity
        {"name": "prefill T=2048 skewed", "kind": "prefill", "tokens": 2048, "hidden": 2048,
         "inter": 512, "experts": 256, "topk": 8, "zipf": 1.1, "residual": False},
        # its router: f16 activations, f32 router weights
        {"name": "router T=2048", "kind": "router", "tokens": 2048, "hidden": 2048,
         "experts": 256, "topk": 8, "f32": False},
        # a long prompt through several layers: the most work in one call
        {"name": "prefill stack T=16384", "kind": "prefill_stack", "layers": 4, "tokens": 16384,
         "hidden": 2048, "inter": 512, "experts": 256, "topk": 8},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["fc", "lm_head", "decode_block", "decode_plan", "routed_plan",
                       "routed_stack", "prefill", "prefill", "run_layer", "run_layer", "fused_op",
                       "router", "prefill_stack"])
    if kind == "fc":
        return {"kind": kind, "k": rng.choice([512, 1024, 2048, 4096]),
                "rows": ",".join(str(_log_int(rng, 1, 8192)) for _ in range(rng.randint(1, 4))),
                "group": rng.choice([32, 64, 128, 256])}
    if kind == "lm_head":
        return {"kind": kind, "k": rng.choice([1024, 2048, 4096]),
                "rows": _log_int(rng, 20001, 248320) // rng.choice([1, 2]), "group": 128,
                "topk": rng.choice([1, 4, 8, 16])}
    if kind == "decode_block":
        return {"kind": kind, "hidden": rng.choice([512, 1024, 2048, 4096]),
                "inter": rng.choice([256, 512, 1024]), "experts": _log_int(rng, 16, 256),
                "group": rng.choice([64, 128]), "topk": rng.choice([1, 2, 4, 8])}
    if kind in ("decode_plan", "routed_plan"):
        return {"kind": kind, "layers": rng.randint(1, 40 if kind == "decode_plan" else 4),
                "hidden": 2048, "inter": 512, "experts": _log_int(rng, 16, 256),
                "group": rng.choice([64, 128, 128]), "topk": rng.randint(1, 8)}
    if kind == "routed_stack":
        return {"kind": kind, "layers": rng.randint(1, 4),
                "hidden": rng.choice([512, 1024, 2048]), "inter": rng.choice([128, 256, 512]),
                "experts": _log_int(rng, 16, 256), "group": rng.choice([64, 128]),
                "topk": rng.choice([2, 4, 8])}
    if kind == "router":
        return {"kind": kind, "tokens": _log_int(rng, 1, 8192),
                "hidden": rng.choice([512, 1024, 2048]), "experts": _log_int(rng, 16, 256),
                "topk": rng.choice([2, 4, 8]), "f32": rng.random() < 0.5}
    hidden, inter = rng.choice([(2048, 512), (2048, 512), (1024, 256), (512, 128), (2048, 768)])
    case = {"kind": kind, "tokens": _log_int(rng, 1, 8192), "hidden": hidden, "inter": inter,
            "experts": rng.choice([256, 256, 128, 60]), "topk": rng.choice([2, 4, 8, 8])}
    if kind == "prefill":
        case.update(zipf=rng.choice([0.0, 0.0, 1.1]), residual=rng.random() < 0.5)
    elif kind == "run_layer":
        case.update(pad=rng.randint(0, 3))
    elif kind == "fused_op":
        case.update(shared=rng.random() < 0.5)
    else:
        case.update(layers=rng.randint(2, 4))
    return case


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _seed(seed, part):
    return int(seed) * 100003 + part


def _layer(c, seed, part, split=False):
    return synth.moe_layer(hidden=c["hidden"], inter=c["inter"], experts=c["experts"],
                           group=c.get("group", 128), seed=_seed(seed, part), device=DEV,
                           split=split)


def _matrix(rows, k, group, seed, part):
    return synth.u4_weight(1, rows, k, group, synth.generator(_seed(seed, part), DEV), DEV)


def _routes(logits, k):
    """Top-k routes of f32 logits [T, E]: ids int32, normalized weights float32."""
    p = torch.softmax(logits.double(), -1)
    v, i = torch.topk(p, k, dim=-1)
    return i.int().contiguous(), (v / v.sum(-1, keepdim=True)).float().contiguous()


def prepare(case, seed):
    c, kind = case, case["kind"]
    s = {"case": c, "ws": pkg.Workspace(DEV)}
    if kind == "fc":
        s["w"] = [_matrix(int(n), c["k"], c["group"], seed, 10 + i)
                  for i, n in enumerate(c["rows"].split(","))]
        # the last of several projections is the router's, whose logits are f32
        s["out"] = [torch.float16] * (len(s["w"]) - 1) + [torch.float32]
        s["x"] = synth.activations(1, c["k"], _seed(seed, 1), DEV)[0].contiguous()
    elif kind == "lm_head":
        s["w"] = _matrix(c["rows"], c["k"], c["group"], seed, 10)
        s["x"] = synth.activations(1, c["k"], _seed(seed, 1), DEV)[0].contiguous()
    elif kind in ("decode_block", "decode_plan", "routed_plan", "routed_stack"):
        L = c.get("layers", 1)
        s["layers"] = [_layer(c, seed, 10 + l) for l in range(L)]
        s["x"] = synth.activations(1, c["hidden"], _seed(seed, 1), DEV)[0].contiguous()
        if kind == "decode_plan":
            s["logits"] = synth.router_logits(L, c["experts"], _seed(seed, 2), DEV)
            s["plan"] = pkg.DecodePlan(s["layers"], k=c["topk"])
        else:
            s["routers"] = [_matrix(c["experts"], c["hidden"], c["group"], seed, 200 + l)
                            for l in range(L)]
        if kind == "routed_plan":
            s["plan"] = pkg.DecodePlan(s["layers"], k=c["topk"], routers=s["routers"])
            s["routes"] = s["plan"].route_buffers()
    elif kind == "router":
        x = synth.activations(c["tokens"], c["hidden"], _seed(seed, 1), DEV)
        s["x"] = x.float() if c["f32"] else x
        g = synth.generator(_seed(seed, 2), DEV)
        s["w"] = torch.randn((c["experts"], c["hidden"]), generator=g,
                             device=DEV) / math.sqrt(c["hidden"])
    else:
        T, k, L = c["tokens"], c["topk"], c.get("layers", 1)
        s["layers"] = [_layer(c, seed, 10 + l, split=kind == "fused_op") for l in range(L)]
        s["x"] = synth.activations(T, c["hidden"], _seed(seed, 1), DEV)
        logits = [synth.router_logits(T, c["experts"], _seed(seed, 100 + l), DEV,
                                      zipf_s=c.get("zipf") or None) for l in range(L)]
        if kind == "fused_op":
            s["logits"] = logits[0]
            if not c["shared"]:
                s["x"] = s["x"].float()
        else:
            r = [_routes(lg, k) for lg in logits]
            s["ids"] = torch.stack([i for i, _ in r]) if L > 1 else r[0][0]
            s["w"] = torch.stack([w for _, w in r]) if L > 1 else r[0][1]
        if kind == "run_layer":
            s["x"] = s["x"].float()
            wide = torch.full((T, k + c["pad"]), -1, dtype=torch.int32, device=DEV)
            wide[:, :k] = s["ids"]
            s["ids"] = wide
        if c.get("residual"):
            s["residual"] = synth.activations(T, c["hidden"], _seed(seed, 3), DEV)
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def run(s):
    c, kind = s["case"], s["case"]["kind"]
    if kind == "fc":
        if len(s["w"]) == 1:
            return pkg.matvec_u4(s["x"], s["w"][0], out_dtype=s["out"][0])
        return pkg.matvec_u4_multi(s["x"], s["w"], s["out"])
    if kind == "lm_head":
        return pkg.lm_head_topk(s["x"], s["w"], c["topk"], ws=s["ws"])
    if kind == "decode_block":
        layer = s["layers"][0]
        h = pkg.apply_rms_norm(s["x"], layer.norm_weight, EPS)
        ids, w, logits = pkg.router_fc_topk(h, s["routers"][0], c["topk"])
        return pkg.run_moe_ffn_layer(layer, h, ids, w, residual=s["x"], ws=s["ws"]), ids, w, logits
    if kind == "decode_plan":
        return s["plan"].run(s["x"], router_logits=s["logits"], epsilon=EPS)
    if kind == "routed_plan":
        r = s["routes"]
        out = s["plan"].run(s["x"], routers=s["routers"], epsilon=EPS, route_out=r)
        return out, r.expert_ids, r.weights, r.logits
    if kind == "routed_stack":
        return pkg.moe_stack_decode_routed(s["layers"], s["routers"], s["x"], c["topk"],
                                           epsilon=EPS, ws=s["ws"])
    if kind == "prefill":
        return pkg.grouped_moe_prefill(s["layers"][0], s["x"], s["ids"], s["w"],
                                       residual=s.get("residual"), ws=s["ws"])
    if kind == "run_layer":
        return pkg.grouped_moe_prefill_routed(s["layers"][0], s["x"], s["ids"], s["w"],
                                              expert_used_count=c["topk"], ws=s["ws"])
    if kind == "fused_op":
        return pkg.moe_3gemm_fused_compressed(s["x"], s["logits"], s["layers"][0], c["topk"],
                                              include_shared=c["shared"], ws=s["ws"])
    if kind == "router":
        return pkg.router_gemm_topk(s["x"], s["w"], c["topk"], ws=s["ws"])
    return pkg.moe_stack_prefill(s["layers"], s["x"], s["ids"], s["w"], EPS, ws=s["ws"])


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _u4_bytes(rows, k, group):
    return rows * k // 2 + rows * (k // group) * 2 + rows * (k // group) // 2


def _expert_bytes(c):
    g = c.get("group", 128)
    return (_u4_bytes(2 * c["inter"], c["hidden"], g) + _u4_bytes(c["hidden"], c["inter"], g))


def _active(c):
    """Experts that the routing of c["tokens"] tokens reaches, as expected."""
    T, E, k = c["tokens"], c["experts"], c["topk"]
    if not c.get("zipf"):
        return E * (1.0 - (1.0 - k / E) ** T)
    g = torch.Generator().manual_seed(1)
    p = torch.arange(1, E + 1, dtype=torch.float64).pow(-c["zipf"])
    logits = torch.randn((T, E), generator=g) + torch.log(p / p.sum()).float()
    return float(torch.unique(torch.topk(logits, k, dim=-1).indices).numel())


def work(case):
    c, kind = case, case["kind"]
    if kind in ("fc", "lm_head"):
        rows = [int(n) for n in str(c["rows"]).split(",")]
        b = sum(_u4_bytes(n, c["k"], c["group"]) + 4 * n for n in rows) + 2 * c["k"]
        return {"bytes": b, "flops": 2 * sum(rows) * c["k"]}
    H, E, k = c["hidden"], c["experts"], c["topk"]
    if kind == "router":
        T = c["tokens"]
        return {"bytes": T * H * (4 if c["f32"] else 2) + E * H * 4 + T * E * 4 + T * k * 8,
                "flops": 2 * T * E * H}
    L, I, shared = c.get("layers", 1), c["inter"], 1
    if kind in ("decode_block", "decode_plan", "routed_plan", "routed_stack"):
        b = (k + 1) * _expert_bytes(c) + H * 6
        f = (k + 1) * 6 * H * I
        if kind == "decode_plan":
            b += E * 4
        else:
            b += _u4_bytes(E, H, c["group"]) + E * 4 + k * 8
            f += 2 * E * H
        return {"bytes": L * b + 4 * H, "flops": L * f}
    T = c["tokens"]
    if kind == "run_layer" or (kind == "fused_op" and not c["shared"]):
        shared = 0
    wide = 8 if not shared else 4
    b = L * ((_active(c) + shared) * _expert_bytes(c) + T * k * 8) + T * H * wide
    if c.get("residual"):
        b += 2 * T * H
    if kind == "fused_op":
        b += T * E * 4
    return {"bytes": b, "flops": L * T * (k + shared) * 6 * H * I}


def tolerance(case):
    """About four times the distance from the 64-bit results."""
    kind = case["kind"]
    if kind == "fc":  # one matrix: f32 out (6e-6 off); several: f16 outputs too (2e-4 off)
        return {"rel": 1e-3 if "," in case["rows"] else 2.5e-5}
    if kind == "lm_head":  # f32 logits, 5e-6 off
        return {"rel": 2.5e-5}
    if kind == "router":  # f32 logits, 1e-6 off; near ties among tokens * k picks
        return {"rel": 1e-5, "differ": 1e-3}
    if kind == "decode_block":  # f16 intermediates and output, 8e-4 to 1.1e-3 off
        return {"rel": 4e-3}
    if kind == "decode_plan":  # f16 residual after every layer: 6e-3 off after 40
        return {"rel": 0.02}
    if kind in ("routed_plan", "routed_stack"):  # the routes' weights follow: 1.2e-3 to 4e-3 off
        return {"rel": 0.015}
    if kind == "prefill_stack":  # f16 weights, intermediates and residual: 1.3e-3 off
        return {"rel": 5e-3}
    return {"rel": 2e-3, "differ": 1e-3}  # f16 weights and intermediates: 5e-4 off


# ---------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# ---------------------------------------------------------------------------

def _dequant(w, e=0):
    """Expert e of a U4 weight in float64 [rows, k]."""
    G = w.k // w.group
    q = w.qweight.reshape(w.experts, w.rows, w.k // 2)[e]
    q = torch.stack([q & 15, q >> 4], -1).reshape(w.rows, G, w.group).double()
    z = w.zp.reshape(w.experts, -1)[e]
    z = torch.stack([z & 15, z >> 4], -1).reshape(-1)[:w.rows * G].reshape(w.rows, G, 1).double()
    sc = w.scale.reshape(w.experts, w.rows, G, 1)[e].double()
    return ((q - z) * sc).reshape(w.rows, w.k)


def _expert(x, gate_up, up, down, e):
    gu = _dequant(gate_up, e)
    gate, upw = (gu, _dequant(up, e)) if up is not None else gu.chunk(2, 0)
    g = x @ gate.T
    return ((g * torch.sigmoid(g)) * (x @ upw.T)) @ _dequant(down, e).T


def _moe(layer, x, ids, w, shared=True):
    """x float64 [T, H], ids [T, k], w [T, k] -> float64 [T, H]."""
    out = torch.zeros_like(x)
    if shared:
        sig = torch.sigmoid(x @ layer.shared_gate_vec.double())
        out += sig[:, None] * _expert(x, layer.shared_gate_up, layer.shared_up,
                                      layer.shared_down, 0)
    ids, w = ids.long(), w.double()
    for e in torch.unique(ids).tolist():
        t, r = (ids == e).nonzero(as_tuple=True)
        out.index_add_(0, t, w[t, r][:, None] * _expert(x[t], layer.gate_up, layer.up,
                                                         layer.down, e))
    return out


def _norm(x, weight):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + EPS) * weight.double()


def _routes64(logits, k):
    v, i = torch.topk(torch.softmax(logits, -1), k, dim=-1)
    return i, v / torch.clamp(v.sum(-1, keepdim=True), min=MIN_SUM)


def exact(case, seed):
    c, kind = case, case["kind"]
    s = prepare(c, seed)
    x = s["x"].double()
    if kind == "fc":
        ys = [_dequant(w) @ x for w in s["w"]]
        return ys if len(ys) > 1 else ys[0]
    if kind == "lm_head":
        y = torch.cat([_dequant(pkg.U4Weight(s["w"].qweight[a:a + 16384],
                                             s["w"].scale[a:a + 16384],
                                             s["w"].zp[a * (c["k"] // c["group"]) // 2:
                                                       (min(a + 16384, c["rows"]) *
                                                        (c["k"] // c["group"]) + 1) // 2],
                                             min(16384, c["rows"] - a), c["k"], c["group"])) @ x
                       for a in range(0, c["rows"], 16384)])
        v, i = torch.topk(y, c["topk"])
        return i, v, y
    if kind == "router":
        logits = x @ s["w"].double().T
        i, w = _routes64(logits, c["topk"])
        return i, w, logits
    if kind in ("decode_block", "routed_plan", "routed_stack"):
        r, got = x[None], []
        for layer, router in zip(s["layers"], s["routers"]):
            h = _norm(r, layer.norm_weight)
            logits = h @ _dequant(router).T
            i, w = _routes64(logits, c["topk"])
            r = r + _moe(layer, h, i, w)
            got.append((i[0], w[0], logits[0]))
        i, w, logits = (torch.stack(v) for v in zip(*got))
        if kind == "decode_block":
            return r[0], i[0], w[0], logits[0]
        return (r[0], i, w, logits) if kind == "routed_plan" else (r[0], i, w)
    if kind == "decode_plan":
        ids, w = _routes64(s["logits"].double(), c["topk"])
        r = x[None]
        for l, layer in enumerate(s["layers"]):
            r = r + _moe(layer, _norm(r, layer.norm_weight), ids[l][None], w[l][None])
        return r[0]
    if kind == "prefill":
        y = _moe(s["layers"][0], x, s["ids"], s["w"])
        return y + s["residual"].double() if c["residual"] else y
    if kind == "run_layer":
        return _moe(s["layers"][0], x, s["ids"][:, :c["topk"]], s["w"], shared=False)
    if kind == "fused_op":
        i, w = _routes64(s["logits"].double(), c["topk"])
        return _moe(s["layers"][0], x, i, w, shared=c["shared"]), i, w
    for l, layer in enumerate(s["layers"]):
        x = x + _moe(layer, _norm(x, layer.norm_weight), s["ids"][l], s["w"][l])
    return x
