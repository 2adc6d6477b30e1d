"""Performance cases of the routed MoE layer: the calls that a program built on
this package makes, over the sizes, formats and batch shapes it meets.

Each case is a dict of plain values. ``kind`` names the entry point:

  layer     ops.MoELayer.forward: router, top-k, experts, shared expert, residual
  stack     ops.MoEStack.forward: consecutive layers with their RMSNorm
  moe       ops.gguf_moe: routed experts with the caller's own routing
  shared    ops.q8_0_gate_up_swiglu + ops.q8_0_matvec_add2: the Q8_0 shared
            expert by itself, added to two residual rows
  norm      ops.NormRouter: RMSNorm, router logits and top-k of decode tokens

Weights are N(0, 0.02) quantised to their GGUF format, activations N(0, 1);
widths are those of the package's own configurations, or generic multiples of
256 (the super-block width).
"""
import math

import numpy as np
import torch

from inferno_amd import BF16, F32, Q2_K, Q3_K, Q4_K, Q6_K, Q8_0, SCORE_SIGMOID, SCORE_SOFTMAX  # noqa: F401
from inferno_amd import ops

QUANT = {"q2k": Q2_K, "q3k": Q3_K, "q4k": Q4_K, "q6k": Q6_K, "q8": Q8_0}
# (values, bytes) of a block
BLOCK = {"q2k": (256, 84), "q3k": (256, 110), "q4k": (256, 144), "q6k": (256, 210),
         "q8": (32, 34)}
EPS = 1e-6

# The four layer shapes of the package's configurations.
SMALL = dict(hidden=2048, experts=64, inter=768, top_k=8, score="softmax", scale=1.0,
             quant="q4k", down="q4k", shared=0, shared_quant="q8", shared_down="q8", x="f32")
XS = dict(SMALL, down="q6k", shared=768, shared_quant="q4k", shared_down="q6k")
GLM = dict(hidden=6144, experts=256, inter=2048, top_k=8, score="sigmoid", scale=2.5,
           quant="q2k", down="q2k", shared=2048, shared_quant="q8", shared_down="q8", x="bf16")
LAGUNA = dict(hidden=4096, experts=128, inter=1536, top_k=10, score="softmax", scale=1.0,
              quant="q2k", down="q2k", shared=1536, shared_quant="q8", shared_down="q8",
              x="bf16")


def _case(kind, shape, tokens, name=None, **more):
    c = dict(shape, kind=kind, tokens=tokens, **more)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the router half of one decode token, in one launch: pure latency
        _case("norm", XS, 1, "norm_router_t1"),
        # one decode token of the smallest layer: launches and latency
        _case("layer", SMALL, 1, "small_t1"),
        # one decode token of the large Q2_K layer with its shared expert
        _case("layer", GLM, 1, "glm_q2k_t1"),
        # one decode token through four layers with their RMSNorms
        _case("stack", LAGUNA, 1, "stack4_t1", layers=4),
        # a few sequences decoded together, or a speculated run of tokens
        _case("layer", GLM, 4, "glm_q2k_t4"),
        # the caller routes (its own top-k or an offloaded router), batched decode
        _case("moe", SMALL, 16, "moe_q4k_t16"),
        # widths off every tuned one, an odd batch
        _case("layer", dict(hidden=2816, experts=96, inter=1280, top_k=6, score="softmax",
                            scale=1.0, quant="q4k", down="q4k", shared=1280, shared_quant="q8",
                            shared_down="q8", x="bf16"), 13, "odd_q4k_t13"),
        # the Q8_0 shared expert of a decode batch, through its own entry points
        _case("shared", GLM, 16, "shared_q8_t16"),
        # a full decode batch of the layer whose shared expert has K-quant formats
        _case("layer", XS, 64, "xs_t64"),
        # batched decode of the Q3_K layer
        _case("layer", dict(LAGUNA, quant="q3k", down="q3k"), 32, "laguna_q3k_t32"),
        # a prompt (or a chunk of one): every expert's weights are read
        _case("layer", dict(GLM, quant="q3k", down="q3k"), 512, "glm_q3k_t512"),
        # the largest prompt chunk: matrix-core work
        _case("layer", GLM, 4096, "glm_q2k_t4096"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    most = work(_case("layer", GLM, 4096))["flops"]
    while True:
        family = rng.choice(["small", "xs", "glm", "laguna", "generic", "generic"])
        if family == "generic":
            q = rng.choice(["q2k", "q3k", "q4k"])
            inter = 256 * rng.randint(2, 9)
            shared = rng.choice([0, inter, 256 * rng.randint(2, 8)])
            sq = rng.choice(["q8", "q8", q])
            down = "q6k" if q == "q4k" and rng.random() < 0.3 else q
            c = dict(hidden=256 * rng.randint(4, 26), experts=rng.randint(16, 256), inter=inter,
                     top_k=rng.randint(2, 10), score=rng.choice(["softmax", "sigmoid"]),
                     scale=rng.choice([1.0, 2.5]), quant=q, down=down, shared=shared,
                     shared_quant=sq, shared_down="q8" if sq == "q8" else down,
                     x=rng.choice(["bf16", "f32"]))
        else:
            c = dict({"small": SMALL, "xs": XS, "glm": GLM, "laguna": LAGUNA}[family])
            if family in ("glm", "laguna"):
                c["quant"] = c["down"] = rng.choice(["q2k", "q3k"])
        kind = rng.choice(["layer"] * 7 + ["moe"] * 2 + ["shared", "stack", "norm"])
        if kind == "stack":
            c = _case("stack", c, rng.randint(1, 4), layers=rng.randint(2, 4))
        elif kind == "norm":
            c = _case("norm", c, rng.randint(1, 16))
        elif kind == "shared":
            c = _case("shared", dict(c, shared=c["shared"] or c["inter"], shared_quant="q8",
                                     shared_down="q8"), _log_int(rng, 1, 512))
        else:
            c = _case(kind, c, _log_int(rng, 1, 4096 if kind == "layer" else 2048))
        if work(c)["flops"] <= most:
            return c


# ------------------------------------------------------------------ inputs

def _normal(g, *shape, std=1.0, dtype=torch.float32):
    return (torch.randn(*shape, generator=g, device="cuda") * std).to(dtype)


def _weights(seed, part, quant, rows, cols):
    return ops.synth_quantized(QUANT[quant], (seed << 8) | part, 0.02, rows, cols)


def _make_layer(c, seed, g, index=0):
    H, E, I, S = c["hidden"], c["experts"], c["inter"], c["shared"]
    p = 16 * index
    t = dict(router=_normal(g, E, H, std=0.02),
             bias=_normal(g, E, std=0.1) if c["score"] == "sigmoid" else None,
             gate=_weights(seed, p, c["quant"], E * I, H),
             up=_weights(seed, p + 1, c["quant"], E * I, H),
             down=_weights(seed, p + 2, c["down"], E * H, I),
             norm=1.0 + _normal(g, H, std=0.1))
    if S:
        t.update(_make_shared(c, seed, p))
    return t


def _make_shared(c, seed, p=0):
    H, S = c["hidden"], c["shared"]
    return dict(sgate=_weights(seed, p + 3, c["shared_quant"], S, H),
                sup=_weights(seed, p + 4, c["shared_quant"], S, H),
                sdown=_weights(seed, p + 5, c["shared_down"], H, S))


def _layer_handle(c, t):
    return ops.MoELayer(
        hidden=c["hidden"], experts=c["experts"], intermediate=c["inter"], top_k=c["top_k"],
        quant=QUANT[c["quant"]], down_quant=QUANT[c["down"]],
        score_fn=SCORE_SIGMOID if c["score"] == "sigmoid" else SCORE_SOFTMAX,
        norm_topk_prob=True, routed_scaling_factor=c["scale"], router=t["router"],
        router_bias=t["bias"], gate=t["gate"], up=t["up"], down=t["down"],
        shared_intermediate=c["shared"], shared_gate=t.get("sgate"), shared_up=t.get("sup"),
        shared_down=t.get("sdown"), shared_quant=QUANT[c["shared_quant"]],
        shared_down_quant=QUANT[c["shared_down"]], max_tokens=c["tokens"])


def _caller_routing(c, g):
    """Distinct experts per token, some more popular than others, in the order
    of their weights; the weights sum to the routing scale."""
    T, E, k = c["tokens"], c["experts"], c["top_k"]
    logit = _normal(g, T, E) + _normal(g, E, std=0.3)
    top = logit.topk(k, dim=1)
    return (top.indices.to(torch.int32).reshape(-1).contiguous(),
            (torch.softmax(top.values, dim=1) * c["scale"]).reshape(-1).contiguous())


def prepare(case, seed):
    c = case
    seed = int(seed)
    g = torch.Generator(device="cuda").manual_seed(seed)
    T, H = c["tokens"], c["hidden"]
    dt = torch.bfloat16 if c["x"] == "bf16" else torch.float32
    s = {"case": c}
    if c["kind"] == "stack":
        s["layers"] = [_make_layer(c, seed, g, l) for l in range(c["layers"])]
        s["x"] = _normal(g, T, H)
        s["handle"] = ops.MoEStack([_layer_handle(c, t) for t in s["layers"]],
                                   [t["norm"] for t in s["layers"]], eps=EPS, act_dtype=dt,
                                   max_tokens=T)
    elif c["kind"] == "layer":
        s["layer"] = _make_layer(c, seed, g)
        s["x"], s["residual"] = _normal(g, T, H, dtype=dt), _normal(g, T, H)
        s["handle"] = _layer_handle(c, s["layer"])
    elif c["kind"] == "moe":
        s["layer"] = _make_layer(dict(c, shared=0), seed, g)
        s["x"] = _normal(g, T, H, dtype=dt)
        s["ids"], s["weights"] = _caller_routing(c, g)
    elif c["kind"] == "shared":
        s["layer"] = _make_shared(c, seed)
        s["x"] = _normal(g, T, H, dtype=dt)
        s["a"], s["b"] = _normal(g, T, H), _normal(g, T, H)
    else:
        s["layer"] = dict(router=_normal(g, c["experts"], H, std=0.02),
                          bias=_normal(g, c["experts"], std=0.1) if c["score"] == "sigmoid" else None,
                          norm=1.0 + _normal(g, H, std=0.1))
        s["x"] = _normal(g, T, H)
        s["handle"] = ops.NormRouter(max_tokens=T)
    return s


def run(state):
    s, c = state, state["case"]
    if c["kind"] == "stack":
        return s["handle"].forward(s["x"])
    if c["kind"] == "layer":
        return s["handle"].forward(s["x"], s["residual"])
    t = s["layer"]
    if c["kind"] == "moe":
        return ops.gguf_moe(QUANT[c["quant"]], QUANT[c["down"]], t["gate"], t["up"], t["down"],
                            s["x"], s["ids"], s["weights"], c["top_k"], c["experts"], c["inter"])
    if c["kind"] == "shared":
        h = ops.q8_0_gate_up_swiglu(t["sgate"], t["sup"], s["x"], c["shared"])
        return h, ops.q8_0_matvec_add2(t["sdown"], h, s["a"], s["b"], c["hidden"])
    normed, logits, ids, w = s["handle"](
        s["x"], t["norm"], EPS, t["router"], t["bias"], c["top_k"],
        SCORE_SIGMOID if c["score"] == "sigmoid" else SCORE_SOFTMAX, True, c["scale"])
    return {"normed": normed, "logits": logits, "ids": ids, "weights": w}


# -------------------------------------------------------------------- work

def _matrix_bytes(quant, rows, cols):
    v, b = BLOCK[quant]
    return rows * cols // v * b


def _experts_used(c):
    """Experts that a batch selects, for router logits of independent normals."""
    T, E, k = c["tokens"], c["experts"], c["top_k"]
    r = np.random.default_rng(7)
    if c["kind"] == "moe":
        key = r.standard_normal((T, E)) + 0.3 * r.standard_normal(E)
    else:
        key = 0.02 * math.sqrt(c["hidden"]) * r.standard_normal((T, E))
        if c["score"] == "sigmoid":
            key = 1.0 / (1.0 + np.exp(-key)) + 0.1 * r.standard_normal(E)
    return len(np.unique(np.argpartition(-key, k - 1, axis=1)[:, :k]))


def work(case):
    c = case
    T, H, E, I, k, S = (c[n] for n in ("tokens", "hidden", "experts", "inter", "top_k", "shared"))
    xb = 2 if c["x"] == "bf16" else 4
    router = 4 * E * H
    shared = (2 * _matrix_bytes(c["shared_quant"], S, H) +
              _matrix_bytes(c["shared_down"], H, S)) if S else 0
    if c["kind"] == "norm":
        return {"bytes": router + 4 * H + T * (8 * H + 4 * E + 8 * k), "flops": 2 * T * H * E}
    if c["kind"] == "shared":
        return {"bytes": shared + T * (xb * H + 8 * S + 12 * H), "flops": 6 * T * H * S}
    one = 2 * _matrix_bytes(c["quant"], I, H) + _matrix_bytes(c["down"], H, I)
    experts, flops = _experts_used(c) * one, 6 * T * k * H * I
    if c["kind"] == "moe":
        return {"bytes": experts + T * (xb * H + 4 * H + 8 * k), "flops": flops}
    flops += 6 * T * H * S + 2 * T * H * E
    if c["kind"] == "layer":
        return {"bytes": experts + shared + router + T * H * (xb + 8), "flops": flops}
    n = c["layers"]
    return {"bytes": n * (experts + shared + router + 4 * H) + 8 * T * H, "flops": n * flops}


# ------------------------------------------------------------------ results

def tolerance(case):
    """About four times what the paths show against 64 bits. The f16 rounding of
    the dequantised weights and of h bounds the layers (the residual, of the
    size of one activation, is part of the output and dilutes it); a stack
    carries each layer's rounding, and the activations' own type, through the
    next; the other two kinds keep 32-bit sums throughout."""
    kind = case["kind"]
    if kind == "norm":
        return {"rel": 1e-6, "max": 1e-5, "differ": 0.01}
    if kind == "shared":
        return {"rel": 1e-5, "max": 1e-4}
    if kind == "stack":
        return {"rel": 8e-3, "max": 0.2}
    if kind == "layer" and case["scale"] == 1.0:
        return {"rel": 1e-3, "max": 0.04}
    return {"rel": 2e-3, "max": 0.04}


def _f16(lo, hi):
    bits = (lo.to(torch.int32) | (hi.to(torch.int32) << 8)).to(torch.int16)
    return bits.view(torch.float16).double().unsqueeze(1)


def _values(quant, raw, rows, cols):
    """The matrix that GGUF blocks hold, in 64 bits (ggml's block layouts)."""
    v, nb = BLOCK[quant]
    b = raw.view(-1, nb)
    n = b.shape[0]
    dev = b.device
    if quant == "q8":
        d = _f16(b[:, 0], b[:, 1])
        return (d * b[:, 2:].contiguous().view(torch.int8).double()).view(rows, cols)
    shift2 = torch.tensor([0, 2, 4, 6], dtype=torch.uint8, device=dev).view(1, 1, 4, 1)
    if quant == "q2k":
        d, dmin = _f16(b[:, 80], b[:, 81]), _f16(b[:, 82], b[:, 83])
        q = (b[:, 16:80].reshape(n, 2, 1, 32) >> shift2) & 3
        sc, mn = d * (b[:, :16] & 15), dmin * (b[:, :16] >> 4)
        w = sc.unsqueeze(2) * q.reshape(n, 16, 16) - mn.unsqueeze(2)
    elif quant == "q3k":
        d = _f16(b[:, 108], b[:, 109])
        low = (b[:, 32:96].reshape(n, 2, 1, 32) >> shift2) & 3
        bit = torch.arange(8, dtype=torch.uint8, device=dev).view(1, 2, 4, 1)
        high = (b[:, :32].reshape(n, 1, 1, 32) >> bit) & 1
        q = (low + 4 * high).double() - 4
        s = b[:, 96:108]
        lo4 = torch.cat([s[:, :8] & 15, s[:, :8] >> 4], 1)
        hi2 = torch.cat([(s[:, 8:] >> (2 * i)) & 3 for i in range(4)], 1)
        w = (d * ((lo4 | (hi2 << 4)).double() - 32)).unsqueeze(2) * q.reshape(n, 16, 16)
    elif quant == "q4k":
        d, dmin = _f16(b[:, 0], b[:, 1]), _f16(b[:, 2], b[:, 3])
        s, qs = b[:, 4:16], b[:, 16:].reshape(n, 4, 1, 32)
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
        q = torch.cat([qs & 15, qs >> 4], 2).reshape(n, 8, 32)
        w = (d * sc).unsqueeze(2) * q - (dmin * mn).unsqueeze(2)
    else:  # q6k
        d = _f16(b[:, 208], b[:, 209])
        ql, qh = b[:, :128].reshape(n, 2, 2, 32), b[:, 128:192].reshape(n, 2, 1, 32)
        low = torch.cat([ql & 15, ql >> 4], 2)
        q = (low | (((qh >> shift2) & 3) << 4)).double() - 32
        sc = d * b[:, 192:208].contiguous().view(torch.int8).double()
        w = sc.unsqueeze(2) * q.reshape(n, 16, 16)
    return w.reshape(rows, cols)


def _ffn(x, quant, down_quant, gate, up, down, inter):
    H = x.shape[1]
    a = x @ _values(quant, gate, inter, H).T
    h = a * torch.sigmoid(a) * (x @ _values(quant, up, inter, H).T)
    return h, h @ _values(down_quant, down, H, inter).T


def _routed(c, t, x, ids, w):
    H, E, I, k = c["hidden"], c["experts"], c["inter"], c["top_k"]
    out = torch.zeros_like(x)
    gate, up, down = (t[n].view(E, -1) for n in ("gate", "up", "down"))
    for e in torch.unique(ids).tolist():
        at = (ids == e).nonzero()
        _, y = _ffn(x[at[:, 0]], c["quant"], c["down"], gate[e], up[e], down[e], I)
        out.index_add_(0, at[:, 0], y * w[at[:, 0], at[:, 1]].unsqueeze(1))
    return out


def _route(c, t, x):
    logits = x @ t["router"].double().T
    bias = 0.0 if t["bias"] is None else t["bias"].double()
    score = torch.sigmoid(logits) if c["score"] == "sigmoid" else logits
    ids = (score + bias).topk(c["top_k"], dim=1).indices
    w = score.gather(1, ids)
    w = w / w.sum(1, keepdim=True) if c["score"] == "sigmoid" else torch.softmax(w, 1)
    return logits, ids, w * c["scale"]


def _norm(x, w):
    return x * torch.rsqrt(x.square().mean(1, keepdim=True) + EPS) * w.double()


def _layer(c, t, x, residual):
    _, ids, w = _route(c, t, x)
    out = residual + _routed(c, t, x, ids, w)
    if c["shared"]:
        out = out + _ffn(x, c["shared_quant"], c["shared_down"], t["sgate"], t["sup"],
                         t["sdown"], c["shared"])[1]
    return out


def exact(case, seed):
    c = case
    s = prepare(case, seed)
    x = s["x"].double()
    if c["kind"] == "stack":
        for t in s["layers"]:
            act = _norm(x, t["norm"]).float()  # the activations' own type is the caller's choice
            x = _layer(c, t, (act.bfloat16() if c["x"] == "bf16" else act).double(), x)
        return x
    t = s["layer"]
    if c["kind"] == "layer":
        return _layer(c, t, x, s["residual"].double())
    if c["kind"] == "moe":
        k = c["top_k"]
        return _routed(c, t, x, s["ids"].view(-1, k), s["weights"].view(-1, k).double())
    if c["kind"] == "shared":
        h, y = _ffn(x, "q8", "q8", t["sgate"], t["sup"], t["sdown"], c["shared"])
        return h, s["a"].double() + s["b"].double() + y
    normed = _norm(x, t["norm"])
    logits, _, w = _route(c, t, normed)
    return {"normed": normed, "logits": logits, "ids": None, "weights": w.reshape(-1)}
