"""The work that programs have this library do, as cases that can be timed.

Four kinds, after the calls of a session that decodes and prefills a
quantized mixture-of-experts model:

  moe      the MoE layers of a decode step: `tokens` = 1 is one sequence, 4 a
           verify window of one token and three drafts, up to 16 a batch of
           sequences.  ``MoeLayer.forward`` on fp32 buffers with the logits
           in hand, or, on the session's fp16 buffers, the router GEMV
           (``gemv_f32_out_f16x``) and ``MoeLayer.forward_f16``.
  prefill  one MoE layer of a prefill chunk, the same two ways through
           ``MoePrefill``.
  proj     a layer's dense projections: Q8_K of the normed activations, the
           two or three input projections, Q8_K of the mixer's output, the
           output projection (added into the residual for one token).
  head     Q8_K of the last hidden states and the LM head, Q4_K or Q6_K.

A decode step's layers are captured into one HIP graph when the program is
set up and replayed each step, as the session does (`graph`); the other
calls are made one by one.  Every layer has weights, inputs and outputs of
its own.  Weights are random blocks whose scales give the dequantized values
the spread of a trained projection (standard deviation about 0.03, mean near
0), activations are N(0, 1) as after a norm.
"""
import math

import torch

from sager_amd import Q4K_BYTES, Q8K_BYTES, ops

Q6K_BYTES = 210
QK = 256

# hidden, n_ff, experts, top-k of the model shape the library's benchmark runs
MODEL = {"hidden": 2048, "n_ff": 512, "experts": 256, "top_k": 8}
# a generic smaller one: super-block counts that are no power of two, an
# expert count that is none either, an odd top-k
OTHER = {"hidden": 1280, "n_ff": 768, "experts": 60, "top_k": 7}


def listed():
    return [
        # one layer, called from the host with nothing captured: what a lone call costs
        {"name": "moe_t1_call", "kind": "moe", **MODEL, "tokens": 1, "layers": 1, "dtype": "f32",
         "shared": True, "gate": False, "sigma": 1.0, "graph": False},
        # the MoE part of one decoded token: 40 layers on the session's buffers
        {"name": "moe_t1_stack", "kind": "moe", **MODEL, "tokens": 1, "layers": 40,
         "dtype": "f16", "shared": True, "gate": True, "sigma": 1.0, "graph": True},
        # the verify window of speculative decoding: a token and three drafts
        {"name": "moe_t4_window", "kind": "moe", **MODEL, "tokens": 4, "layers": 10,
         "dtype": "f16", "shared": True, "gate": True, "sigma": 1.5, "graph": True},
        # thirteen sequences decoded together
        {"name": "moe_t13_batch", "kind": "moe", **MODEL, "tokens": 13, "layers": 4,
         "dtype": "f32", "shared": True, "gate": False, "sigma": 1.0, "graph": True},
        # a short prompt
        {"name": "prefill_t57", "kind": "prefill", **MODEL, "tokens": 57, "dtype": "f16",
         "shared": True, "gate": True, "sigma": 1.0},
        # the ragged last chunk of a prompt, another model shape, no shared expert
        {"name": "prefill_t509", "kind": "prefill", **OTHER, "tokens": 509, "dtype": "f32",
         "shared": False, "gate": False, "sigma": 1.0},
        # the benchmark's prefill chunk on the session's buffers
        {"name": "prefill_t2048", "kind": "prefill", **MODEL, "tokens": 2048, "dtype": "f16",
         "shared": True, "gate": True, "sigma": 1.0},
        # a long chunk on fp32 buffers, the largest
        {"name": "prefill_t4096", "kind": "prefill", **MODEL, "tokens": 4096, "dtype": "f32",
         "shared": True, "gate": False, "sigma": 1.0},
        # the dense projections of one decoded token, 40 layers
        {"name": "proj_t1_stack", "kind": "proj", "hidden": 2048, "mixer": 4096, "tokens": 1,
         "layers": 40, "graph": True},
        # the same of a window of six tokens
        {"name": "proj_t6_window", "kind": "proj", "hidden": 2048, "mixer": 4096, "tokens": 6,
         "layers": 20, "graph": True},
        # the head as model files hold it, one token
        {"name": "head_q6_t1", "kind": "head", "format": "q6", "rows": 248320, "hidden": 2048,
         "tokens": 1},
        # the logits of a verify window from a Q4_K head
        {"name": "head_q4_t4", "kind": "head", "format": "q4", "rows": 248320, "hidden": 2048,
         "tokens": 4},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["moe", "moe", "prefill", "prefill", "proj", "head"])
    if kind in ("moe", "prefill"):
        shape = dict(MODEL) if rng.random() < 0.6 else {
            "hidden": rng.choice([768, 1280, 2048, 3072]), "n_ff": rng.choice([512, 768, 1024]),
            "experts": rng.choice([32, 60, 128, 200]), "top_k": rng.choice([4, 6, 7, 8])}
        f16 = rng.random() < 0.6
        shared = rng.random() < 0.7
        case = {"kind": kind, **shape, "dtype": "f16" if f16 else "f32", "shared": shared,
                "gate": shared and rng.random() < 0.5, "sigma": rng.choice([1.0, 1.5])}
        if kind == "moe":
            # (the layer holds Q8_K of every slot's h in one workgroup's LDS)
            blocks = (shape["top_k"] + 1) * shape["n_ff"] // QK
            tokens = _log_int(rng, 1, min(16, 320 // blocks))
            per_layer = 3 * (shape["experts"] + 1) * shape["hidden"] * shape["n_ff"] * 9 // 16
            most = max(2, min(24, int(7e9) // per_layer, 64 // tokens))
            return {**case, "tokens": tokens, "layers": rng.randint(2, most), "graph": True}
        scale = MODEL["hidden"] * MODEL["n_ff"] / (shape["hidden"] * shape["n_ff"])
        return {**case, "tokens": _log_int(rng, 17, int(4000 * min(1.0, scale)))}
    if kind == "proj":
        tokens = _log_int(rng, 1, 16)
        return {"kind": "proj", "hidden": rng.choice([1024, 2048, 2304]),
                "mixer": rng.choice([2048, 4096]), "tokens": tokens,
                "layers": rng.randint(4, max(5, 40 // tokens)), "graph": True}
    if rng.random() < 0.4:
        return {"kind": "head", "format": "q6", "rows": _log_int(rng, 20000, 248320),
                "hidden": rng.choice([1280, 2048]), "tokens": 1}
    tokens = _log_int(rng, 1, 16)
    return {"kind": "head", "format": "q4",
            "rows": _log_int(rng, 20000, 248320 if tokens <= 4 else 100000),
            "hidden": rng.choice([1280, 2048]), "tokens": tokens}


# ---- inputs -------------------------------------------------------------------

def _generator(seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 1000003 + salt)
    return g


def _random_bytes(n, gen):
    v = torch.empty((n + 7) // 8, dtype=torch.int64, device="cuda")
    v.random_(-2 ** 63, 2 ** 63 - 1, generator=gen)
    return v.view(torch.uint8)[:n]


def _q4(rows, k, gen):
    """Random Q4_K blocks [rows * k/256, 144]: uniform quants and 6-bit
    scales/mins, d near 1.5e-4 and dmin near 7.5 d, so that the weights
    d*sc*q - dmin*mn have a mean near 0."""
    n = rows * k // QK
    b = _random_bytes(n * Q4K_BYTES, gen).view(n, Q4K_BYTES)
    d = 1.5e-4 * (0.5 + torch.rand((n, 1), device="cuda", generator=gen))
    m = 7.5 * d * (0.8 + 0.4 * torch.rand((n, 1), device="cuda", generator=gen))
    b[:, :4] = torch.cat([d, m], 1).half().view(torch.uint8)
    return b


def _q6(rows, k, gen):
    """Random Q6_K blocks [rows * k/256, 210], d near 2e-5."""
    n = rows * k // QK
    b = _random_bytes(n * Q6K_BYTES, gen).view(n, Q6K_BYTES)
    d = 2e-5 * (0.5 + torch.rand((n, 1), device="cuda", generator=gen))
    b[:, 208:] = d.half().view(torch.uint8)
    return b


def _normal(gen, *shape, scale=1.0, dtype=torch.float32):
    return (torch.randn(shape, device="cuda", generator=gen) * scale).to(dtype)


def _proj_rows(case, layer):
    """Rows of a layer's input projections: every fourth layer has q | k | v,
    the others the two of a gated linear mixer."""
    m = case["mixer"]
    return (m, m // 8, m // 8) if layer % 4 == 3 else (2 * m, 64)


def _inputs(case, seed):
    """Weights and activations of a case, from the seed alone."""
    kind, T, H = case["kind"], case["tokens"], case["hidden"]
    if kind == "head":
        gen = _generator(seed, 4)
        make = _q6 if case["format"] == "q6" else _q4
        return {"w": make(case["rows"], H, gen), "x": _normal(gen, T, H, dtype=torch.float16)}
    if kind == "proj":
        layers = []
        for i in range(case["layers"]):
            gen = _generator(seed, 100 + i)
            rows = _proj_rows(case, i)
            layers.append({
                "rows": rows, "w_in": [_q4(r, H, gen) for r in rows],
                "w_out": _q4(H, case["mixer"], gen),
                "xn": _normal(gen, T, H, dtype=torch.float16),
                "mixed": _normal(gen, T, case["mixer"], scale=0.1, dtype=torch.float16),
                "residual": _normal(gen, T, H, dtype=torch.float16)})
        return layers
    F, E = case["n_ff"], case["experts"]
    act = torch.float16 if case["dtype"] == "f16" else torch.float32
    layers = []
    for i in range(case.get("layers", 1)):
        gen = _generator(seed, 1000 + i)
        n = E + 1 if case["shared"] else E
        layer = {"experts": _q4(3 * n * F, H, gen).view(3, n, -1),
                 "x": _normal(gen, T, H, dtype=act),
                 "residual": _normal(gen, T, H, dtype=act),
                 "gate_w": _normal(gen, H, scale=0.03) if case["gate"] else None}
        if case["dtype"] == "f16":
            layer["router"] = _normal(gen, E, H, scale=case["sigma"] / math.sqrt(H))
        else:
            layer["logits"] = _normal(gen, T, E, scale=case["sigma"])
        layers.append(layer)
    return layers


# ---- the calls ----------------------------------------------------------------

def _moe_layer(case, layer):
    """What a program keeps for one MoE layer: pointer tables, the layer
    object with its workspace, output buffers."""
    E, T, H, k = case["experts"], case["tokens"], case["hidden"], case["top_k"]
    w = layer["experts"]
    at = torch.arange(E, dtype=torch.int64, device="cuda") * w.shape[2]
    tabs = [(at + w[m, 0].data_ptr()).contiguous() for m in range(3)]
    shared = tuple(w[m, E] for m in range(3)) if case["shared"] else None
    make = ops.MoeLayer if case["kind"] == "moe" else ops.MoePrefill
    return make(*tabs, shared, hidden=H, n_ff=case["n_ff"], n_expert=E, k=k, max_tokens=T,
                shared_gate_w=layer["gate_w"])


def _moe_pass(case, state):
    for i, layer in enumerate(state["inputs"]):
        obj = state["objects"][i]
        out, idx, weight = state["out"][i], state["idx"][i], state["weight"][i]
        if case["dtype"] == "f16":
            logits = ops.gemv_f32_out_f16x(layer["router"], layer["x"], y=state["logits"][i])
            obj.forward_f16(layer["x"], logits=logits, residual=layer["residual"], out=out,
                            idx=idx, weight=weight)
        else:
            obj.forward(layer["x"], layer["logits"], residual=layer["residual"], out=out,
                        idx=idx, weight=weight)


def _proj_pass(case, state):
    H, M, T = case["hidden"], case["mixer"], case["tokens"]
    for layer, buf in zip(state["inputs"], state["buffers"]):
        xq = ops.quantize_q8_k(layer["xn"], out=buf["xq"])
        if T == 1:
            ops.gemv_nm_q4_k_q8_f16out(layer["w_in"], xq, layer["rows"], H, ys=buf["y_in"])
        else:
            for w, r, y in zip(layer["w_in"], layer["rows"], buf["y_in"]):
                ops.gemv_q4_k_q8_f16out_batched(w, xq, r, H, T, y=y)
        mq = ops.quantize_q8_k(layer["mixed"], out=buf["mq"])
        if T == 1:
            ops.gemv_q4_k_q8_f16out_resadd(layer["w_out"], mq, layer["residual"], H, M,
                                           y=buf["y_out"])
        else:
            ops.gemv_q4_k_q8_f16out_batched(layer["w_out"], mq, H, M, T, y=buf["y_out"])


def _captured(case, state, one_pass):
    """One pass captured into a HIP graph, after a pass on other residuals
    (the library loads its kernels on first use)."""
    kept = [layer["residual"].clone() for layer in state["inputs"]]
    one_pass(case, state)
    for layer, r in zip(state["inputs"], kept):
        layer["residual"].copy_(r)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        one_pass(case, state)
    return graph


def prepare(case, seed):
    inputs = _inputs(case, seed)
    state = {"case": case, "inputs": inputs}
    T, H = case["tokens"], case["hidden"]
    if case["kind"] == "head":
        state["xq"] = ops.q8k_empty(T, H)
        state["y"] = torch.empty((T, case["rows"]), device="cuda")
        return state
    L = len(inputs)
    if case["kind"] == "proj":
        def f16(*shape):
            return torch.empty(shape, dtype=torch.float16, device="cuda")
        state["y_in"] = f16(T * sum(sum(layer["rows"]) for layer in inputs))
        state["y_out"] = f16(L, T, H)
        state["residual"] = torch.stack([layer["residual"] for layer in inputs])
        state["buffers"], at = [], 0
        for i, layer in enumerate(inputs):
            layer["residual"] = state["residual"][i]
            ys = []
            for r in layer["rows"]:
                ys.append(state["y_in"][at:at + r * T].view(T, r))
                at += r * T
            state["buffers"].append({"xq": ops.q8k_empty(T, H),
                                     "mq": ops.q8k_empty(T, case["mixer"]),
                                     "y_in": ys, "y_out": state["y_out"][i]})
        one_pass = _proj_pass
    else:
        act = torch.float16 if case["dtype"] == "f16" else torch.float32
        k = case["top_k"]
        state["objects"] = [_moe_layer(case, layer) for layer in inputs]
        state["out"] = torch.zeros((L, T, H), dtype=act, device="cuda")
        state["idx"] = torch.full((L, T, k + 1), -1, dtype=torch.int32, device="cuda")
        state["weight"] = torch.zeros((L, T, k + 1), device="cuda")
        if case["dtype"] == "f16":
            state["logits"] = torch.zeros((L, T, case["experts"]), device="cuda")
        one_pass = _moe_pass
    if case.get("graph"):
        state["graph"] = _captured(case, state, one_pass)
    else:
        state["pass"] = one_pass
    return state


def run(state):
    case, inputs = state["case"], state["inputs"]
    if case["kind"] == "head":
        T, rows, H = case["tokens"], case["rows"], case["hidden"]
        xq = ops.quantize_q8_k(inputs["x"], out=state["xq"])
        y = state["y"]
        if case["format"] == "q6":
            ops.gemv_q6_k_q8(inputs["w"], xq, rows, H, y=y)
        elif T == 1:
            ops.gemv_q4_k_q8(inputs["w"], xq, rows, H, y=y)
        else:
            ops.gemv_q4_k_q8_batched(inputs["w"], xq, rows, H, T, y=y)
        return {"logits": y}
    if "graph" in state:
        state["graph"].replay()
    else:
        state["pass"](case, state)
    if case["kind"] == "proj":
        out = {"y_in": state["y_in"], "y_out": state["y_out"]}
        if case["tokens"] == 1:
            out["residual"] = state["residual"]
        return out
    out = {"out": state["out"], "idx": state["idx"][..., :case["top_k"]],
           "weight": state["weight"]}
    if case["dtype"] == "f16":
        out["logits"] = state["logits"]
    return out


# ---- what a pass cannot do without --------------------------------------------

def work(case):
    T, H = case["tokens"], case["hidden"]
    if case["kind"] == "head":
        n = case["rows"] * H
        per_block = Q6K_BYTES if case["format"] == "q6" else Q4K_BYTES
        return {"bytes": n / QK * per_block + 2 * T * H + 4 * T * case["rows"],
                "flops": 2.0 * T * n}
    if case["kind"] == "proj":
        total = flops = 0
        for i in range(case["layers"]):
            rows, M = sum(_proj_rows(case, i)), case["mixer"]
            n = rows * H + H * M
            total += n / QK * Q4K_BYTES + 2 * T * (H + rows + M + H + (2 * H if T == 1 else 0))
            flops += 2.0 * T * n
        return {"bytes": total, "flops": flops}
    F, E, k = case["n_ff"], case["experts"], case["top_k"]
    touched = E * (1 - (1 - k / E) ** T) + (1 if case["shared"] else 0)
    slots = k + (1 if case["shared"] else 0)
    act = 2 if case["dtype"] == "f16" else 4
    one = touched * 3 * H * F / QK * Q4K_BYTES + 3 * T * H * act + 4 * T * E + 8 * T * (k + 1)
    flops = 6.0 * T * slots * H * F
    if case["dtype"] == "f16":
        one += 4 * E * H
        flops += 2.0 * T * E * H
    layers = case.get("layers", 1)
    return {"bytes": layers * one, "flops": layers * flops}


# From the error against exact(), measured over listed and drawn cases.  What
# moves the results of a correct implementation of a layer is not its sums but
# the 8-bit codes of h inside it: a change of one fp32 rounding moves a code by
# one where h/d lies near a half (f32 buffers: up to 2.1e-4 seen), and so do
# the fp16 roundings of g, u and h, which exact() does not make (f16 buffers:
# 2.1e-3 to 2.9e-3).  The projections round fp32 row sums to fp16 (2.3e-4 to
# 3.5e-4), the head's fp32 row sums are within 1e-7.
def tolerance(case):
    if case["kind"] == "head":
        return {"rel": 1e-6}
    if case["kind"] == "proj":
        return {"rel": 1e-3}
    return {"rel": 5e-3 if case["dtype"] == "f16" else 1e-3, "differ": 1e-3}


# ---- the same in 64 bits ------------------------------------------------------

def _weights_q4(b, rows, k):
    """Q4_K blocks -> fp64 [rows, k]."""
    b = b.reshape(-1, Q4K_BYTES)
    n = b.shape[0]
    dd = b[:, :4].contiguous().view(torch.float16).double()
    s = b[:, 4:16].to(torch.int32)
    sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double()
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
    q = b[:, 16:].reshape(n, 4, 1, 32)
    q = torch.cat([q & 15, q >> 4], 2).reshape(n, 8, 32).double()
    w = (dd[:, 0:1] * sc)[:, :, None] * q - (dd[:, 1:2] * mn)[:, :, None]
    return w.reshape(rows, k)


def _weights_q6(b, rows, k):
    """Q6_K blocks -> fp64 [rows, k]."""
    b = b.reshape(-1, Q6K_BYTES)
    n = b.shape[0]
    d = b[:, 208:].contiguous().view(torch.float16).double()
    sc = b[:, 192:208].contiguous().view(torch.int8).double()
    lo = b[:, :128].reshape(n, 2, 2, 32).to(torch.int32)
    hi = b[:, 128:192].reshape(n, 2, 32).to(torch.int32)
    q = torch.stack([(lo[:, :, j % 2] >> (4 * (j // 2)) & 15) | ((hi >> (2 * j) & 3) << 4)
                     for j in range(4)], 2)
    q = (q - 32).double().reshape(n, 16, 16)
    return (d[:, :, None] * sc[:, :, None] * q).reshape(rows, k)


def _q8(x):
    """What Q8_K keeps of x's rows: codes times d, per 256 values."""
    v = x.double().reshape(-1, QK)
    d = v.abs().amax(1, keepdim=True).clamp_min(1e-30) / 127
    return ((v / d).round().clamp(-127, 127) * d).reshape(x.shape)


def _exact_moe(case, layer):
    T, H, F, E, k = (case[n] for n in ("tokens", "hidden", "n_ff", "experts", "top_k"))
    x = layer["x"].double()
    if case["dtype"] == "f16":
        logits = x @ layer["router"].double().T
    else:
        logits = layer["logits"].double()
    p, idx = torch.softmax(logits, 1).topk(k, dim=1)
    weight = torch.cat([p / p.sum(1, keepdim=True), torch.ones((T, 1), device="cuda").double()], 1)
    xq = _q8(x)
    out = layer["residual"].double()

    def expert(e, rows):
        w = [_weights_q4(layer["experts"][m, e], *s) for m, s in ((0, (F, H)), (1, (F, H)),
                                                                  (2, (H, F)))]
        g, u = xq[rows] @ w[0].T, xq[rows] @ w[1].T
        return _q8(g / (1 + torch.exp(-g)) * u) @ w[2].T

    used = torch.unique(idx).tolist()
    for e in used:
        rows, slot = torch.nonzero(idx == e, as_tuple=True)
        out.index_add_(0, rows, expert(e, rows) * weight[rows, slot][:, None])
    if case["shared"]:
        y = expert(E, torch.arange(T, device="cuda"))
        if case["gate"]:
            y = y * torch.sigmoid(x @ layer["gate_w"].double())[:, None]
        out = out + y
    return out, weight, logits


def exact(case, seed):
    inputs = _inputs(case, seed)
    if case["kind"] == "head":
        xq, H, step = _q8(inputs["x"]), case["hidden"], 16384
        per_row = H // QK
        decode = _weights_q6 if case["format"] == "q6" else _weights_q4
        parts = [xq @ decode(inputs["w"][a * per_row:min(a + step, case["rows"]) * per_row],
                             min(step, case["rows"] - a), H).T
                 for a in range(0, case["rows"], step)]
        return {"logits": torch.cat(parts, 1)}
    if case["kind"] == "proj":
        H, M = case["hidden"], case["mixer"]
        y_in, y_out = [], []
        for layer in inputs:
            xq, mq = _q8(layer["xn"]), _q8(layer["mixed"])
            y_in += [(xq @ _weights_q4(w, r, H).T).reshape(-1)
                     for w, r in zip(layer["w_in"], layer["rows"])]
            y_out.append(mq @ _weights_q4(layer["w_out"], H, M).T)
        out = {"y_in": torch.cat(y_in), "y_out": torch.stack(y_out)}
        if case["tokens"] == 1:
            out["residual"] = torch.stack([layer["residual"].double() + y
                                           for layer, y in zip(inputs, y_out)])
        return out
    got = [_exact_moe(case, layer) for layer in inputs]
    out = {"out": torch.stack([g[0] for g in got]), "idx": None,
           "weight": torch.stack([g[1] for g in got])}
    if case["dtype"] == "f16":
        out["logits"] = torch.stack([g[2] for g in got])
    return out
