"""The measured workloads of the MoE feed-forward path, through its public entry points.

Every case is the SF37 layer shape (288 experts, top-8, 4096 x 1280, Q3GU gate/up and Q2D down
experts, a shared expert), which is the shape the engine and every BASELINE configuration run; what
varies is what varies in use: tokens per call (1 for a decode step, 2-16 for a batch of sequences,
tens for larger batches and draft verification, hundreds to thousands for prefill chunks), layers per
call, how tokens spread over the experts, the router's and the shared expert's format, and the caller
(the layer call, the layer stack, or the engine's own sequence of mapped entry points).

A case's fields:
  entry    "layer": sf37_hip_moe_layer; "stack": sf37_hip_moe_stack (norm, layer, residual per layer);
           "engine": the engine's per-layer branch (libsf37_engine_moe.so) over a registered model map
  tokens   rows per call
  layers   independently seeded layers run one after the other in a pass (weights of several layers
           keep a decode pass from being served by the 256 MB cache, as a model's 45 layers do)
  routing  "router": logits computed from the rows; "zipf": injected logits N(0, 1) with a per-expert
           popularity bias of Zipf exponent 1.1 (configs.zipf_bias), the skew of real prefill traffic
  router   "f32", "bf16" or "q8_0" router weights (the engine's dense types)
  shared   "q8_0" (the engine's shared expert) or "q3q2" (the same formats as the routed experts)
  il       layer index of the first layer: 43 and 44 clamp the SwiGLU
"""
from __future__ import annotations

import ctypes as C
import math
import os

import numpy as np
import torch

from sf37_amd import configs, hip, moe

E, D, F, K = moe.EXPERTS, moe.EMBD, moe.EXPERT_FF, moe.EXPERT_USED
EPS, SCALE = 1e-5, 3.0
EXPERT_BYTES = 2 * F * (D // 256) * 110 + D * (F // 256) * 84
ROUTER_BYTES = {"f32": E * D * 4, "bf16": E * D * 2, "q8_0": E * (D // 32) * 34}
SHARED_BYTES = {"q8_0": 3 * D * F // 32 * 34, "q3q2": EXPERT_BYTES}
ROUTER_TYPE = {"f32": hip.TYPE_F32, "bf16": hip.TYPE_BF16, "q8_0": hip.TYPE_Q8_0}
DEV = "cuda"


def _case(name, entry, tokens, layers=1, routing="router", router="f32", shared="q8_0", il=10):
    c = {"entry": entry, "tokens": tokens, "layers": layers, "routing": routing, "router": router,
         "shared": shared, "il": il}
    return dict(c, name=name) if name else c


def listed():
    return [
        # one generated token through consecutive layers: latency and launches (config 4's decode)
        _case("decode_1", "stack", 1, layers=6),
        # the same through the engine's branch: a dozen small calls per layer
        _case("engine_decode_1", "engine", 1, layers=4),
        # a small serving batch (config 1)
        _case("decode_8", "layer", 8, layers=2),
        # the largest fused decode batch, shared expert in the routed formats, the clamped last layers
        _case("decode_16_q3q2", "stack", 16, layers=2, shared="q3q2", il=43),
        # just past the fused decode batch: a larger serving batch, or draft tokens being verified
        _case("batch_21", "layer", 21),
        # a large serving batch, popular experts shared by many rows
        _case("batch_64_zipf", "layer", 64, routing="zipf", router="q8_0"),
        # a short prompt of odd length, bf16 router, shared expert in the routed formats
        _case("prompt_187", "layer", 187, router="bf16", shared="q3q2"),
        # a medium prefill chunk under skewed routing (config 2)
        _case("prefill_512_zipf", "layer", 512, routing="zipf"),
        # an odd prompt through the engine's branch
        _case("engine_prefill_777", "engine", 777, router="q8_0"),
        # a long chunk through two layers with norm and residual, skewed routing (config 4's prefill)
        _case("stack_2048_zipf", "stack", 2048, layers=2, routing="zipf"),
        # the largest chunk, even routing (config 3)
        _case("prefill_4096", "layer", 4096),
    ]


def draw(rng):
    entry = rng.choice(["layer", "layer", "stack", "engine"])
    most = {"layer": 4096, "stack": 2048, "engine": 1536}[entry]
    tokens = min(most, int(math.exp(rng.uniform(0.0, math.log(most + 1)))))
    layers = rng.randint(3, 6) if tokens == 1 else 2 if tokens <= 16 else 1
    routing = "router" if entry == "engine" else rng.choice(["router", "router", "zipf"])
    router = rng.choice(["f32", "f32", "q8_0"] if entry == "engine" else ["f32", "f32", "bf16", "q8_0"])
    shared = "q8_0" if entry == "engine" else rng.choice(["q8_0", "q8_0", "q3q2"])
    return _case(None, entry, tokens, layers, routing, router, shared, rng.randint(3, 45 - layers))


# ---- inputs --------------------------------------------------------------------------------------

class _Map:
    """torch's view of a library tensor (the tensor lives as long as the view)."""

    def __init__(self, t, shape, typestr):
        self.t = t
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "data": (t.device_ptr(), False),
                                         "version": 2}


def _torch(t, shape, dtype=torch.float32):
    typestr = {torch.float32: "<f4", torch.int32: "<i4", torch.uint8: "|u1"}[dtype]
    return torch.as_tensor(_Map(t, shape, typestr), device=DEV)


def _bytes(t):
    return _torch(t, (t.nbytes,), torch.uint8)


_KEYS = []      # model-map keys (host addresses that stay unique while the process lives)


def _register(parts):
    """A model map whose ranges are the given device tensors: (key address, size, {name: offset})."""
    key = np.zeros(64, np.uint8)
    _KEYS.append(key)
    off, pos = {}, 0
    size = sum(t.nbytes + 256 for t in parts.values())
    for name, t in parts.items():
        off[name] = pos
        hip.check(hip.lib().sf37_hip_register_device_range(key.ctypes.data, size, pos, t.nbytes, t.h), "register")
        pos = (pos + t.nbytes + 255) // 256 * 256
    return key.ctypes.data, size, off


def _layer(case, seed, l):
    """One synthetic layer with its router in the case's format and bf16 norm weights."""
    il = case["il"] + l
    s = moe.layer_seed(seed, il)
    lay = moe.SynthLayer(s, il=il, shared=case["shared"])
    f32 = _torch(lay.router, (E, D))
    if case["router"] == "bf16":
        router = hip.Tensor.alloc(E * D * 2)
        _bytes(router).copy_(f32.to(torch.bfloat16).view(torch.uint8).reshape(-1))
    elif case["router"] == "q8_0":
        router = hip.synth_quant("q8_0", E, D, s, 9)
    else:
        router = lay.router
    norm = hip.Tensor.alloc(D * 2)
    g = torch.Generator(DEV).manual_seed(s)
    _bytes(norm).copy_((torch.randn(D, generator=g, device=DEV) * 0.02).to(torch.bfloat16).view(torch.uint8).reshape(-1))
    w = lay.weights_struct(SCALE)
    w.router, w.router_type = router.h, ROUTER_TYPE[case["router"]]
    return {"lay": lay, "router": router, "norm": norm, "struct": w}


def _inputs(case, seed):
    hip.init()
    T, n = case["tokens"], case["layers"]
    ls = [_layer(case, seed, l) for l in range(n)]
    x = hip.synth_normal(T * D, seed, configs.X_STREAM)
    logits = None
    if case["routing"] == "zipf":
        g = torch.Generator(DEV).manual_seed(seed)
        logits = []
        for l in range(n):
            t = hip.empty((T, E), np.float32)
            bias = torch.from_numpy(configs.zipf_bias(moe.layer_seed(seed, l))).to(DEV)
            _torch(t, (T, E)).copy_(torch.randn(T, E, generator=g, device=DEV) + bias)
            logits.append(t)
    return {"case": dict(case), "layers": ls, "x": x, "logits": logits}


class _EngineLayer(C.Structure):
    _fields_ = [("map", C.c_void_p), ("size", C.c_uint64), ("il", C.c_uint32), ("router_type", C.c_uint32)] + \
        [(f, C.c_uint64) for f in ("post_norm", "router_gate", "router_bias", "share_gate", "share_up", "share_down",
                                   "moe_gate", "moe_up", "moe_down")] + \
        [(f, C.c_uint32) for f in ("n_expert", "topk", "embd", "expert_ff")]


_BUFS = ("hidden", "ffn_norm", "gate", "up", "mid", "ffn_out", "router_logits", "router_probs", "router_selected",
         "router_weights", "routed_gate", "routed_up", "routed_mid", "routed_down", "routed_out")


class _EngineBufs(C.Structure):
    _fields_ = [(n, C.c_void_p) for n in _BUFS]


def _engine():
    L = C.CDLL(os.path.join(hip.PKG, "libsf37_engine_moe.so"))
    L.sf37_engine_moe_decode.argtypes = [C.POINTER(_EngineLayer), C.POINTER(_EngineBufs)]
    L.sf37_engine_moe_prefill.argtypes = [C.POINTER(_EngineLayer), C.POINTER(_EngineBufs), C.c_uint32]
    return L


def prepare(case, seed):
    s = _inputs(case, seed)
    T, n = case["tokens"], case["layers"]
    sel = [hip.empty((T, K), np.int32) for _ in range(n)]
    s["sel"] = sel
    outputs = {"selected": [_torch(t, (T, K), torch.int32) for t in sel]}
    if case["entry"] == "layer":
        s["out"] = [hip.empty((T, D), np.float32) for _ in range(n)]
        s["wts"] = [hip.empty((T, K), np.float32) for _ in range(n)]
        outputs["out"] = [_torch(t, (T, D)) for t in s["out"]]
        outputs["weights"] = [_torch(t, (T, K)) for t in s["wts"]]
    elif case["entry"] == "stack":
        s["h"] = hip.empty((T, D), np.float32)
        key, size, off = _register({"norm%d" % l: d["norm"] for l, d in enumerate(s["layers"])})
        Ta = C.c_void_p * n
        s["stack"] = ((hip.LayerWeights * n)(*[d["struct"] for d in s["layers"]]), key, size,
                      (C.c_uint64 * n)(*[off["norm%d" % l] for l in range(n)]),
                      Ta(*[t.h for t in s["logits"]]) if s["logits"] else None, Ta(*[t.h for t in sel]))
        outputs["hidden"] = _torch(s["h"], (T, D))
    else:
        s["engine"], s["engine_layers"] = _engine(), []
        R = max(T, K)
        shapes = {"hidden": T * D, "ffn_norm": T * D, "gate": R * F, "up": R * F, "mid": R * F, "ffn_out": T * D,
                  "router_logits": T * E, "router_probs": T * E, "router_weights": T * K, "routed_gate": T * K * F,
                  "routed_up": T * K * F, "routed_mid": T * K * F, "routed_down": K * D, "routed_out": T * D}
        s["bufs"] = {k: hip.empty(v, np.float32) for k, v in shapes.items()}
        s["logits_out"] = [hip.empty((T, E), np.float32) for _ in range(n)]
        s["engine_bufs"] = []
        for l, d in enumerate(s["layers"]):
            lay = d["lay"]
            key, size, off = _register({"norm": d["norm"], "router": d["router"], "bias": lay.router_bias,
                                        "sg": lay.sh_gate, "su": lay.sh_up, "sd": lay.sh_down, "g": lay.gate,
                                        "u": lay.up, "d": lay.down})
            s["engine_layers"].append(_EngineLayer(
                key, size, lay.il, ROUTER_TYPE[case["router"]], off["norm"], off["router"], off["bias"], off["sg"],
                off["su"], off["sd"], off["g"], off["u"], off["d"], E, K, D, F))
            bufs = dict(s["bufs"], router_selected=sel[l], router_logits=s["logits_out"][l])
            s["engine_bufs"].append(_EngineBufs(*[bufs[k].h for k in _BUFS]))
        outputs["hidden"] = _torch(s["bufs"]["hidden"], (T, D))
        outputs["logits"] = [_torch(t, (T, E)) for t in s["logits_out"]]
    s["outputs"] = outputs
    hip.synchronize()
    return s


def run(state):
    case, L = state["case"], hip.lib()
    T, n = case["tokens"], case["layers"]
    if case["entry"] == "layer":
        for l in range(n):
            lg = state["logits"][l].h if state["logits"] else None
            hip.check(L.sf37_hip_moe_layer(state["out"][l].h, state["sel"][l].h, state["wts"][l].h,
                                           state["layers"][l]["struct"], lg, state["x"].h, T), "moe_layer")
        return state["outputs"]
    hidden = state["h"] if case["entry"] == "stack" else state["bufs"]["hidden"]
    hip.check(L.sf37_hip_tensor_copy(hidden.h, 0, state["x"].h, 0, T * D * 4), "copy of the rows")
    if case["entry"] == "stack":
        structs, key, size, offs, lg, sel = state["stack"]
        hip.check(L.sf37_hip_moe_stack(hidden.h, n, structs, key, size, offs, EPS, lg, sel, T), "moe_stack")
    else:
        for l in range(n):
            a = (C.byref(state["engine_layers"][l]), C.byref(state["engine_bufs"][l]))
            ok = state["engine"].sf37_engine_moe_decode(*a) if T == 1 else \
                state["engine"].sf37_engine_moe_prefill(*a, T)
            hip.check(ok, "engine layer")
    return state["outputs"]


# ---- what a pass cannot do without, and how close two correct answers are -----------------------

def work(case):
    T, n = case["tokens"], case["layers"]
    total = 0
    for l in range(n):
        rng = np.random.default_rng([T, l])
        lg = rng.standard_normal((T, E))
        if case["routing"] == "zipf":
            lg = lg + configs.zipf_bias(l)[None, :]
        distinct = np.unique(np.argpartition(-lg, K - 1, axis=1)[:, :K]).size
        total += distinct * EXPERT_BYTES + ROUTER_BYTES[case["router"]] + SHARED_BYTES[case["shared"]]
        total += T * E * 4 if case["routing"] == "zipf" else 0
        if case["entry"] == "layer":
            total += 2 * T * D * 4          # the rows in, the output out
    if case["entry"] != "layer":
        total += 2 * T * D * 4              # a chain of layers reads its rows once and writes them once
    return {"bytes": total, "flops": n * T * (2 * 3 * D * F * (K + 1) + 2 * D * E)}


def tolerance(case):
    """A layer quantises its rows and each expert's hidden row to 8-bit codes: a sum in another order
    moves such a row by an ulp, which now and then moves a code by one, and in a chain of layers the
    next layer's rows and codes with it.  Measured against exact() over several seeds: up to 1.8e-4 for
    one layer, 1.1e-3 with the norm before it (its rows then differ by ulps too), 4.4e-3 through two
    layers, 2.4e-2 through four to six (one token, where a single code is a visible share of a row);
    about four times that is stated.  Selected experts differ only where scores (nearly) tie: one
    swapped pair in a chain."""
    chain = case["entry"] != "layer"
    rel = 7e-4 if not chain else 4e-3 if case["layers"] == 1 else 2e-2 if case["layers"] == 2 else 1e-1
    return {"rel": rel, "differ": max(1e-3, 2.0 / (case["tokens"] * K)) if chain else 1e-3}


# ---- the path in 64 bits -------------------------------------------------------------------------

def _f16(b):
    return b.contiguous().view(torch.float16).double()


def _deq_q8_0(raw, rows, cols):
    b = raw.reshape(rows, cols // 32, 34)
    return (_f16(b[..., :2]) * b[..., 2:].contiguous().view(torch.int8).double()).reshape(rows, cols)


def _deq_low(raw, rows, cols, bits):
    """Blocks of 256: four f16 scales, four zero points, four groups of 64 codes of 3 or 2 bits."""
    size = 110 if bits == 3 else 84
    b = raw.reshape(rows, cols // 256, size)
    s = _f16(b[..., :8]).unsqueeze(-1)
    zp = (b[..., 8:12] & (7 if bits == 3 else 3)).double().unsqueeze(-1)
    p = b[..., 12:12 + 32 * bits].to(torch.int32)
    if bits == 3:
        t = p.reshape(rows, cols // 256, 32, 3)
        word = t[..., 0] | t[..., 1] << 8 | t[..., 2] << 16
        q = torch.stack([word >> (3 * k) & 7 for k in range(8)], -1)
    else:
        q = torch.stack([p >> (2 * k) & 3 for k in range(4)], -1)
    return ((q.reshape(rows, cols // 256, 4, 64).double() - zp) * s).reshape(rows, cols)


def _codes(x, block):
    """The rows after 8-bit block quantisation (scale = max / 127), as the formats define it."""
    b = x.float().reshape(x.shape[0], -1, block)
    d = b.abs().amax(-1, keepdim=True) / 127.0
    inv = torch.where(d > 0, 1.0 / d, torch.zeros_like(d))
    return (torch.round(b * inv).clamp(-128, 127).double() * d.double()).reshape(x.shape[0], -1)


def _swiglu(g, u, w, clamp):
    if clamp > 1e-6:
        g, u = g.clamp(max=clamp), u.clamp(-clamp, clamp)
    return g * torch.sigmoid(g) * u * w


def _exact_layer(case, d, x, logits):
    """(out, selected, weights, logits) of one layer on rows x (float32)."""
    lay, T = d["lay"], x.shape[0]
    xb = x.double()
    if case["router"] == "q8_0":
        mine = _codes(x, 32) @ _deq_q8_0(_bytes(d["router"]), E, D).T
    elif case["router"] == "bf16":
        mine = xb @ _bytes(d["router"]).view(torch.bfloat16).reshape(E, D).double().T
    else:
        mine = xb @ _torch(d["router"], (E, D)).double().T
    lg = mine.float() if logits is None else logits
    p = torch.sigmoid(lg.double())
    score = p.float() + _torch(lay.router_bias, (E,))
    order = torch.sort(score, dim=1, descending=True, stable=True).indices[:, :K]
    pk = torch.gather(p, 1, order)
    wts = pk / pk.sum(1, keepdim=True).clamp(min=1e-20) * SCALE
    x8 = _codes(x, 256)
    pairs = torch.zeros(T * K, D, dtype=torch.float64, device=DEV)
    flat, wflat = order.reshape(-1), wts.reshape(-1)
    gb, db = F * lay.g_row, D * lay.d_row
    gate, up, down = _bytes(lay.gate), _bytes(lay.up), _bytes(lay.down)
    for e in torch.unique(flat).tolist():
        at = torch.nonzero(flat == e).reshape(-1)
        rows = x8[at // K]
        g = rows @ _deq_low(gate[e * gb:(e + 1) * gb], F, D, 3).T
        u = rows @ _deq_low(up[e * gb:(e + 1) * gb], F, D, 3).T
        mid = _codes(_swiglu(g, u, wflat[at].unsqueeze(1), lay.clamp_routed), 256)
        pairs[at] = mid @ _deq_low(down[e * db:(e + 1) * db], D, F, 2).T
    out = pairs.reshape(T, K, D).sum(1)
    if case["shared"] == "q3q2":
        deq, xs, block = (lambda t, r, c, b: _deq_low(_bytes(t), r, c, b)), x8, 256
    else:
        deq, xs, block = (lambda t, r, c, b: _deq_q8_0(_bytes(t), r, c)), _codes(x, 32), 32
    mid = _swiglu(xs @ deq(lay.sh_gate, F, D, 3).T, xs @ deq(lay.sh_up, F, D, 3).T, 1.0, lay.clamp_shared)
    out = out + _codes(mid, block) @ deq(lay.sh_down, D, F, 2).T
    return out, order.int(), wts, mine


def exact(case, seed):
    """The formats' arithmetic in binary64: rows and hidden rows quantised as the formats say, the products and
    everything else in 64 bits."""
    s = _inputs(case, seed)
    hip.synchronize()
    x = _torch(s["x"], (case["tokens"], D))
    r = {"selected": []}
    lg = [_torch(t, (case["tokens"], E)) for t in s["logits"]] if s["logits"] else [None] * case["layers"]
    if case["entry"] == "layer":
        r["out"], r["weights"] = [], []
        for d, l in zip(s["layers"], lg):
            out, sel, wts, _ = _exact_layer(case, d, x, l)
            r["out"].append(out)
            r["selected"].append(sel)
            r["weights"].append(wts)
        return r
    h = x.double()
    logits = []
    for d, l in zip(s["layers"], lg):
        w = _bytes(d["norm"]).view(torch.bfloat16).double()
        xn = h / torch.sqrt((h * h).mean(1, keepdim=True) + EPS) * (1.0 + w)
        out, sel, _, mine = _exact_layer(case, d, xn.float(), l)
        h = h + out
        r["selected"].append(sel)
        logits.append(mine)
    r["hidden"] = h
    if case["entry"] == "engine":
        r["logits"] = logits
    return r
