"""The MoE-layer calls that decide how fast a model runs on this library: what is timed, and what it must return.

A case is one pass of a program through the public entry points:
    entry "routed"   experts.run_routed: router, routed (and merged shared) experts and the residual of one block
    entry "variant"  variants.hip_*.run(state, x, idx, wts): the experts on ids that the caller has routed
A case with graph = True runs `layers` such calls as one captured HIP graph (experts.reserve, backend.capture), as a
decode loop replays its steps; every layer reads its own activations, as a block reads what its attention wrote. The
others are eager calls of one layer.

Shapes are the model shapes of shapes.py, or generic ones. Weights are bell-shaped around zero, as a quantiser leaves
them: 4-bit codes with a scale per group (int4 g64: scale and bias in bf16; MXFP4: an E8M0 byte per 32), expert biases
where the model has them. Activations and router weights are normal; skew "zipf" adds a Zipf(1.1) popularity to the
router's logits.
"""
import importlib
import math

import numpy as np
import torch

import __graft_entry__

__graft_entry__.load_package()
experts = importlib.import_module("moelab_amd.experts")
backend = importlib.import_module("moelab_amd.backend")
SHAPES = importlib.import_module("moelab_amd.shapes").SHAPES
VARIANT = {("int4", 0): importlib.import_module("moelab_amd.variants.hip_q4_moe"),
           ("int4", 1): importlib.import_module("moelab_amd.variants.hip_q4_moe"),
           ("mxfp4", 0): importlib.import_module("moelab_amd.variants.hip_mxfp4_moe"),
           ("mxfp4", 1): importlib.import_module("moelab_amd.variants.hip_mxfp4_moe"),
           ("mxfp4", 2): importlib.import_module("moelab_amd.variants.hip_mxfp4_gptoss")}

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)
DEV = "cuda"


def _case(name, shape, T, *, fmt="int4", entry="routed", layers=1, graph=False, x="bf16", out=None, act=0,
          biases=False, norm=True, skew="uniform", residual=True):
    s = SHAPES[shape] if isinstance(shape, str) else shape
    d, f, E, k, S = (s.d, s.f, s.E, s.k, s.shared) if isinstance(shape, str) else s
    c = dict(d=d, f=f, E=E, k=k, S=S, T=T, fmt=fmt, entry=entry, layers=layers, graph=graph, x=x, out=out or x,
             act=act, biases=biases, norm=norm, skew=skew, residual=residual)
    return c if name is None else dict(c, name=name)


def listed():
    gpt = dict(fmt="mxfp4", act=2, biases=True)
    return [
        # one token of one sequence: the MoE blocks of a third of a 48-layer model (a pipeline stage), replayed per token
        _case("qwen3_30b decode T1", "qwen3-30b-a3b", 1, layers=16, graph=True),
        # the same on MXFP4 experts with biases, half the model's 24 layers
        _case("gptoss_20b decode T1", "gpt-oss-20b", 1, layers=12, graph=True, **gpt),
        # a single eager call of the smallest size: what a program without graphs sees
        _case("olmoe eager T1", "olmoe-1b-7b", 1, entry="variant", residual=False),
        # checking five drafted tokens at once, ids routed by the caller
        _case("olmoe verify T5", "olmoe-1b-7b", 5, entry="variant", layers=8, graph=True),
        # decode steps of a serving batch: skewed routing, and an odd batch on MXFP4
        _case("qwen3_30b batch T32", "qwen3-30b-a3b", 32, layers=8, graph=True, skew="zipf"),
        _case("gptoss_20b batch T27", "gpt-oss-20b", 27, layers=4, graph=True, **gpt),
        # a large model's decode batch, little shared between tokens
        _case("qwen3_235b batch T64", "qwen3-235b-a22b", 64),
        # a ragged prompt with two shared experts merged into the routed set, greedy gate
        _case("dsv2_lite prompt T237", "deepseek-v2-lite", 237, norm=False),
        # a ragged prompt in half precision, ids routed by the caller
        _case("olmoe fp16 prompt T333", "olmoe-1b-7b", 333, entry="variant", x="fp16"),
        # prefill: prompts on few large experts, in either format, and a chunk of a long prompt on many small ones
        _case("mixtral prefill T512", "mixtral-8x7b", 512),
        _case("gptoss_20b prefill T1500", "gpt-oss-20b", 1500, **gpt),
        _case("qwen3_30b prefill T4096", "qwen3-30b-a3b", 4096, skew="zipf"),
    ]


#: Bounds on a drawn case: floating operations and packed weight bytes of one layer; the largest listed cases have
#: 361e9 (mixtral prefill) and 1.4e9 (qwen3_235b batch).
MAX_FLOPS, MAX_WEIGHTS = 300e9, 1.4e9


def draw(rng):
    """A case of the same ranges: a model's shape or a generic one, T from 1 to 4096, either format, any x dtype."""
    while True:
        if rng.random() < 0.6:
            name = rng.choice(["olmoe-1b-7b", "qwen3-30b-a3b", "gpt-oss-20b", "deepseek-v2-lite", "mixtral-8x7b",
                               "qwen3-235b-a22b"])
            s = SHAPES[name]
            shape = (s.d, s.f, s.E, s.k, s.shared)
            fmt = "mxfp4" if name.startswith("gpt-oss") else rng.choice(["int4", "int4", "int4", "mxfp4"])
        else:
            d, f = (64 * int(round(math.exp(rng.uniform(math.log(a), math.log(b))))) for a, b in ((8, 80), (4, 64)))
            E = rng.choice([8, 16, 24, 32, 60, 64, 128, 160])
            shape = (d, f, E, min(E, rng.randint(1, 8)), 0)
            fmt = rng.choice(["int4", "mxfp4"])
        gpt = fmt == "mxfp4" and rng.random() < 0.6
        T = int(round(math.exp(rng.uniform(0.0, math.log(4096)))))
        x = rng.choice(["bf16", "bf16", "bf16", "bf16", "fp16", "fp32"])
        entry = "routed" if x == "bf16" and rng.random() < 0.7 else "variant"
        graph = T <= 64 and rng.random() < 0.6
        d, f, E, k, S = shape
        c = _case(None, shape if entry == "routed" else (d, f, E, k, 0), T, fmt=fmt, entry=entry, x=x, graph=graph,
                  layers=rng.randint(2, 8) if graph else 1, out="fp32" if rng.random() < 0.15 else x,
                  act=2 if gpt else rng.choice([0, 0, 0, 1]), biases=gpt, norm=rng.random() < 0.7,
                  skew=rng.choice(["uniform", "zipf"]), residual=rng.random() < 0.7)
        if 6.0 * T * (k + c["S"]) * d * f <= MAX_FLOPS and c["layers"] * (E + c["S"]) * _expert_bytes(c) <= MAX_WEIGHTS:
            return c


# ------------------------------------------------------------------------------------------------------- inputs
def _codes(N, K, E, fmt, g):
    """int32 words [E, N, K/8] of bell-shaped 4-bit codes, low nibble first."""
    z = torch.empty((E, N, K), device=DEV).normal_(generator=g)
    if fmt == "int4":
        q = z.mul_(2.5).add_(8.0).round_().clamp_(0, 15).to(torch.uint8)
    else:
        mags = torch.tensor(E2M1, device=DEV)
        neg = (z < 0).to(torch.uint8)
        q = torch.bucketize(z.mul_(2.2).abs_(), (mags[1:] + mags[:-1]) / 2).to(torch.uint8)
        q |= neg << 3
    del z
    return (q[..., 0::2] | (q[..., 1::2] << 4)).contiguous().view(torch.int32)


def _proj(N, K, E, fmt, g):
    """One projection in the reference's layout, its weights about N(0, 1 / K)."""
    codes = _codes(N, K, E, fmt, g)
    if fmt == "int4":
        scales = torch.rand((E, N, K // 64), generator=g, device=DEV).mul_(0.7).add_(0.65).mul_(K ** -0.5 / 2.5)
        scales = scales.to(torch.bfloat16)
        return codes, scales, (scales.float() * -8.0).to(torch.bfloat16)
    e = 127 + int(round(math.log2(K ** -0.5 / 2.2)))
    return codes, torch.randint(e - 1, e + 2, (E, N, K // 32), generator=g, device=DEV).to(torch.uint8)


def _gen(seed, layer):
    return torch.Generator(device=DEV).manual_seed(1000003 * (seed + 1) + layer)


def _weights(c, seed, layer):
    """{g, u, d: packed projections, sg, su, sd: the shared experts', bg, bu, bd, wr, rbias: or None}."""
    g = _gen(seed, layer)
    d, f, E, S, fmt = c["d"], c["f"], c["E"], c["S"], c["fmt"]
    w = {n: _proj(N, K, E, fmt, g) for n, N, K in (("g", f, d), ("u", f, d), ("d", d, f))}
    if S:
        w.update({"s" + n: _proj(N, K, S, fmt, g) for n, N, K in (("g", f, d), ("u", f, d), ("d", d, f))})
    for n, N in (("bg", f), ("bu", f), ("bd", d)):
        w[n] = torch.randn((E, N), generator=g, device=DEV).mul_(0.05).to(torch.bfloat16).float() if c["biases"] else None
    w["wr"] = torch.randn((E, d), generator=g, device=DEV).mul_(0.02).to(torch.bfloat16)
    rb = torch.randn(E, generator=g, device=DEV) * 0.1 if c["biases"] else torch.zeros(E, device=DEV)
    if c["skew"] == "zipf":
        pop = torch.log(torch.arange(1, E + 1, device=DEV).float()) * -1.1
        rb = rb + pop[torch.randperm(E, generator=g, device=DEV)]
    w["rbias"] = rb if c["biases"] or c["skew"] == "zipf" else None
    return w


def _inputs(c, seed, layer):
    """(x [T, d], residual [T, d] or None, idx, wts of the caller's router or None)."""
    g = _gen(seed, layer + 500)
    T, d, E, k = c["T"], c["d"], c["E"], c["k"]
    x = torch.randn((T, d), generator=g, device=DEV).to(DTYPES[c["x"]])
    res = torch.randn((T, d), generator=g, device=DEV).to(DTYPES[c["out"]]) if c["residual"] else None
    if c["entry"] == "routed":
        return x, res, None, None
    logits = torch.randn((T, E), generator=g, device=DEV)
    if c["skew"] == "zipf":
        pop = torch.log(torch.arange(1, E + 1, device=DEV).float()) * -1.1
        logits = logits + pop[torch.randperm(E, generator=g, device=DEV)]
    top, idx = logits.topk(k, dim=1)
    return x, res, idx.to(torch.int32), torch.softmax(top, 1)


def _state(c, w):
    mod = VARIANT[c["fmt"], c["act"]]
    if c["act"] == 2:
        return mod.state(w["g"], w["u"], w["d"], w["bg"], w["bu"], w["bd"])
    s = mod.state_from_packed(w["g"], w["u"], w["d"], w["bg"], w["bu"], w["bd"])
    if c["S"]:
        s["shared"] = mod.state_from_packed(w["sg"], w["su"], w["sd"])
        s = experts.merge_shared(s)
    return s


def _call(c, s, w, x, res, idx, wts, out):
    """One layer through its entry point: {y, and the routing where the call does it}."""
    if c["entry"] == "routed":
        y, idx, wts = experts.run_routed(s, x, w["wr"], c["k"], bias=w["rbias"], norm=c["norm"], act=c["act"],
                                         residual=res, out=out, out_dtype=DTYPES[c["out"]])
        return {"y": y, "idx": idx, "wts": wts}
    mod = VARIANT[c["fmt"], c["act"]]
    kw = {} if c["act"] == 2 else {"act": c["act"]}   # the gpt-oss variant's state holds its activation
    return {"y": mod.run(s, x, idx, wts, residual=res, out_dtype=DTYPES[c["out"]], **kw)}


def prepare(case, seed):
    c = case
    layers = []
    for l in range(c["layers"]):
        w = _weights(c, seed, l)
        s = _state(c, w)
        keep = {"wr": w["wr"], "rbias": w["rbias"]}
        del w
        layers.append((s, keep, *_inputs(c, seed, l), None))
    if not c["graph"]:
        return {"case": c, "layer": layers[0]}
    for layer in layers:
        experts.reserve(layer[0], c["T"], c["k"])
    graph, outs = backend.capture(lambda: [_call(c, *layer) for layer in layers])
    return {"case": c, "layers": layers, "graph": graph, "outs": outs}


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["outs"]
    return _call(state["case"], *state["layer"])


# --------------------------------------------------------------------------------------------- work and tolerance
def _expert_bytes(c):
    return 3 * c["d"] * c["f"] * (0.5625 if c["fmt"] == "int4" else 0.53125)


def _distinct(c):
    """Experts that T tokens select, simulated from the case's popularity."""
    T, E, k = c["T"], c["E"], c["k"]
    rng = np.random.default_rng(7)
    logits = rng.standard_normal((T, E)) * (0.02 * math.sqrt(c["d"]) if c["entry"] == "routed" else 1.0)
    if c["skew"] == "zipf":
        logits -= 1.1 * np.log(np.arange(1, E + 1))
    return len(np.unique(np.argpartition(-logits, k - 1, axis=1)[:, :k]))


def work(case):
    """Every selected expert read once in its packed form, x and the residual once, y written once."""
    c = case
    size = {"bf16": 2, "fp16": 2, "fp32": 4}
    by = (_distinct(c) + c["S"]) * _expert_bytes(c)
    if c["biases"]:
        by += _distinct(c) * 4 * (2 * c["f"] + c["d"])
    by += c["T"] * c["d"] * (size[c["x"]] + size[c["out"]] * (2 if c["residual"] else 1)) + c["T"] * c["k"] * 8
    fl = 6.0 * c["T"] * (c["k"] + c["S"]) * c["d"] * c["f"]
    if c["entry"] == "routed":
        by += 2 * c["E"] * c["d"]
        fl += 2.0 * c["T"] * c["E"] * c["d"]
    return {"bytes": float(c["layers"] * by), "flops": float(c["layers"] * fl)}


def tolerance(case):
    """About four times what the outputs differ from exact(): 1.7e-3 in bf16 and 2.1e-4 in fp16, which is the rounding
    of y, and up to 2.3e-4 in fp32, where operands of 11 to 16 bits (fp16 weights and activations of the dense int4
    tiles, h in two bf16 planes) show. Two roundings of y can lie one step apart; an id may move where two logits tie."""
    rel = {"bf16": 7e-3, "fp16": 1e-3, "fp32": 1e-3}[case["out"]]
    return {"rel": rel, "max": {"bf16": 3e-2, "fp16": 1e-2, "fp32": 1e-2}[case["out"]], "differ": 1e-3}


# ------------------------------------------------------------------------------------------------ 64-bit reference
def _dequant(p, e, fmt):
    """Expert e of one packed projection in float64 [N, K]."""
    b = p[0][e].contiguous().view(torch.uint8)
    q = torch.stack([b & 15, b >> 4], -1).flatten(-2)
    if fmt == "int4":
        return (q.double().unflatten(-1, (-1, 64)) * p[1][e].double()[..., None] + p[2][e].double()[..., None]).flatten(-2)
    v = torch.tensor(E2M1 + tuple(-m for m in E2M1), dtype=torch.float64, device=DEV)[q.long()]
    return (v.unflatten(-1, (-1, 32)) * torch.exp2(p[1][e].double() - 127.0)[..., None]).flatten(-2)


def _glu(g, u, act):
    if act == 2:
        g, u = g.clamp(max=7.0), u.clamp(-7.0, 7.0)
        return g * torch.sigmoid(1.702 * g) * (u + 1.0)
    return (torch.nn.functional.gelu(g, approximate="tanh") if act else torch.nn.functional.silu(g)) * u


def _exact_layer(c, seed, layer):
    w = _weights(c, seed, layer)
    x, res, idx, wts = _inputs(c, seed, layer)
    out, k, x = {}, c["k"], x.double()
    if c["entry"] == "routed":
        logits = x @ w["wr"].double().t()
        if w["rbias"] is not None:
            logits = logits + w["rbias"].double()
        top, idx = logits.topk(k, dim=1)
        wts = torch.softmax(top, 1) if c["norm"] else torch.softmax(logits, 1).gather(1, idx)
        out = {"idx": idx, "wts": wts}
    y = torch.zeros_like(x) if res is None else res.double()
    wts = wts.double()
    for e in range(c["E"]):
        tok, j = (idx == e).nonzero(as_tuple=True)
        if tok.numel():
            xe = x[tok]
            g, u = xe @ _dequant(w["g"], e, c["fmt"]).t(), xe @ _dequant(w["u"], e, c["fmt"]).t()
            if c["biases"]:
                g, u = g + w["bg"][e].double(), u + w["bu"][e].double()
            o = _glu(g, u, c["act"]) @ _dequant(w["d"], e, c["fmt"]).t()
            if c["biases"]:
                o = o + w["bd"][e].double()
            y.index_add_(0, tok, o * wts[tok, j][:, None])
    for e in range(c["S"]):
        g, u = (x @ _dequant(w[n], e, c["fmt"]).t() for n in ("sg", "su"))
        y = y + _glu(g, u, c["act"]) @ _dequant(w["sd"], e, c["fmt"]).t()
    return {"y": y, **out}


def exact(case, seed):
    got = [_exact_layer(case, seed, l) for l in range(case["layers"])]
    return got if case["graph"] else got[0]
