"""The work that programs have this library do, as cases that can be timed: the MoE FFN sublayer from one token to a long
prompt, the hyper-connection mix in front of it, dense quantized projections, and the sublayer's launches with FP32
activations.

Shapes: "wide" is the benchmark's (H 3072, 512 experts, top-10, I 512, Q4 g128, a separate shared Q8 expert), "served"
the served model's (H 2560, I 640, 512 experts + the stacked shared one, top-10, Q4 g128), "small" the benchmark's Q8
model (H 2048, 64 experts, top-8, I 512, Q8 g64, no shared expert). Weights have a standard deviation near 0.02 and
activations near 1, so the shared and the routed experts contribute alike.
"""
import math

import numpy as np
import torch

from strixite_amd import moe

SHAPES = {
    "wide": {"H": 3072, "E": 512, "k": 10, "I": 512, "bits": 4, "G": 128, "shared": "separate"},
    "served": {"H": 2560, "E": 512, "k": 10, "I": 640, "bits": 4, "G": 128, "shared": "stacked"},
    "small": {"H": 2048, "E": 64, "k": 8, "I": 512, "bits": 8, "G": 64, "shared": "none"},
}
LAYERS = 8  # layers of a decode step: independent weights, so that each layer's experts come from HBM


def listed():
    return [
        # one user's decode step, eight layers deep in one graph: launches and latency set the time
        {"name": "decode_1_small", "kind": "stack", "shape": "small", "M": 1},
        {"name": "decode_1_served", "kind": "stack", "shape": "served", "M": 1},
        # two users with seven drafts each (the benchmark's decode step), and a ragged batch of the served model
        {"name": "decode_16_wide", "kind": "stack", "shape": "wide", "M": 16},
        {"name": "decode_11_served", "kind": "stack", "shape": "served", "M": 11},
        # a server's batch: six users with seven drafts each
        {"name": "decode_48_wide", "kind": "stack", "shape": "wide", "M": 48},
        # a short prompt of odd length, evenly routed
        {"name": "prefill_333_served", "kind": "layer", "shape": "served", "M": 333, "zipf": 0.0},
        # a long prompt (one chunk of it) with skewed routing, and the Q8 model's
        {"name": "prefill_4096_wide", "kind": "layer", "shape": "wide", "M": 4096, "zipf": 1.0},
        {"name": "prefill_1500_small", "kind": "layer", "shape": "small", "M": 1500, "zipf": 0.5},
        # the hyper-connection mix around a sublayer: a decode step and a prompt
        {"name": "mix_16", "kind": "mix", "T": 16, "d": 2560, "r": 320, "bits": 4, "G": 64, "act": "bf16"},
        {"name": "mix_2000", "kind": "mix", "T": 2000, "d": 2560, "r": 320, "bits": 4, "G": 64, "act": "bf16"},
        # a dense Q8 FFN through its own calls (projection, SwiGLU, projection) at a ragged batch
        {"name": "dense_100", "kind": "dense", "M": 100, "H": 3072, "I": 512, "bits": 8, "G": 64},
        # the engine's FP32 activation mode: the sublayer launch by launch
        {"name": "f32_40_wide", "kind": "f32", "shape": "wide", "M": 40},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["stack", "stack", "stack", "layer", "layer", "layer", "mix", "mix", "dense", "f32"])
    if kind == "stack":
        return {"kind": kind, "shape": rng.choice(sorted(SHAPES)), "M": _log_int(rng, 1, 64)}
    if kind == "layer":
        return {"kind": kind, "shape": rng.choice(sorted(SHAPES)), "M": _log_int(rng, 65, 4000),
                "zipf": rng.choice([0.0, 0.5, 1.0])}
    if kind == "mix":
        return {"kind": kind, "T": _log_int(rng, 1, 4000), "d": 128 * rng.randint(8, 24), "r": 64 * rng.randint(2, 6),
                "bits": rng.choice([4, 8]), "G": 64, "act": rng.choice(["bf16", "bf16", "f32"])}
    if kind == "dense":
        return {"kind": kind, "M": _log_int(rng, 1, 2000), "H": 256 * rng.randint(6, 16), "I": 128 * rng.randint(3, 16),
                "bits": rng.choice([4, 8]), "G": rng.choice([64, 128])}
    return {"kind": kind, "shape": rng.choice(["wide", "served"]), "M": _log_int(rng, 1, 48)}


# ---- inputs ------------------------------------------------------------------------------------------------------
def _weight(g, bits, N, K, G, std=0.02):
    """Uniform codes with scales around std (times 0.5 .. 1.5) and the min that centres them."""
    n = N * K * bits // 8
    q = torch.randint(-(1 << 63), (1 << 63) - 1, ((n + 7) // 8,), dtype=torch.int64, device="cuda", generator=g)
    levels = (1 << bits) - 1
    s = torch.rand(N * (K // G), device="cuda", generator=g).add_(0.5).mul_(std * math.sqrt(12.0) / (levels + 1))
    s = s.to(torch.bfloat16)
    m = (s.float() * (-0.5 * levels)).to(torch.bfloat16)
    return moe.QWeight(bits, q.view(torch.uint8)[:n], s.view(torch.int16), m.view(torch.int16), N, K, G)


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _layer(g, shape, zipf=0.0):
    c = SHAPES[shape]
    H, E, I, stacked = c["H"], c["E"], c["I"], c["shared"] == "stacked"
    rows = E + (0 if c["shared"] == "none" else 1)
    router = (torch.randn((rows, H), device="cuda", generator=g) * 0.02).to(torch.bfloat16)
    bias = None
    if zipf:
        rank = torch.randperm(E, device="cuda", generator=g).float() + 1.0
        bias = -1.1 * zipf * rank.log()
    Es = E + (1 if stacked else 0)
    gu = _weight(g, c["bits"], Es * 2 * I, H, c["G"])
    dn = _weight(g, c["bits"], Es * H, I, c["G"])
    sgu = sdn = None
    if c["shared"] == "separate":
        sgu, sdn = _weight(g, 8, 2 * I, H, 64), _weight(g, 8, H, I, 64)
    return moe.MoeLayer(H, E, c["k"], I, router, gu, dn, bias, sgu, sdn, shared_stacked=stacked)


def _x(g, M, K, dtype=torch.bfloat16):
    return torch.randn((M, K), device="cuda", generator=g).to(dtype)


def _buffers(layer, M):
    return {"y": torch.empty((M, layer.H), dtype=torch.bfloat16, device="cuda"),
            "x_out": torch.empty((M, layer.H), dtype=torch.bfloat16, device="cuda"),
            "ids": torch.empty((M, layer.A), dtype=torch.int32, device="cuda"),
            "coef": torch.empty((M, layer.A), dtype=torch.float32, device="cuda"),
            "err": torch.zeros(6, dtype=torch.int32, device="cuda")}


def prepare(case, seed):
    g = _gen(seed)
    kind, st = case["kind"], {"case": case}
    if kind == "stack":
        M = case["M"]
        st["layers"] = [_layer(g, case["shape"]) for _ in range(LAYERS)]
        st["x"] = [_x(g, M, L.H) for L in st["layers"]]
        st["ctx"] = moe.LayerContext()
        st["ws"] = st["layers"][0].workspace(M)
        st["out"] = [_buffers(L, M) for L in st["layers"]]

        def step():
            for L, x, out in zip(st["layers"], st["x"], st["out"]):
                L.forward(x, ws=st["ws"], out=out, ctx=st["ctx"])

        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            step()
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        st["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(st["graph"]):
            step()
    elif kind == "layer":
        st["layer"] = _layer(g, case["shape"], case["zipf"])
        st["x"] = _x(g, case["M"], st["layer"].H)
        st["ctx"], st["ws"] = moe.LayerContext(), st["layer"].workspace(case["M"])
        st["out"] = _buffers(st["layer"], case["M"])
    elif kind == "mix":
        d, r = case["d"], case["r"]
        st["x"] = _x(g, case["T"], 4 * d, torch.bfloat16 if case["act"] == "bf16" else torch.float32)
        st["down"] = _weight(g, case["bits"], r + 4, 4 * d, case["G"])
        st["up"] = _weight(g, case["bits"], 4 * d, r, case["G"], 0.05)  # its arrays are chunk-major
        st["norm"] = torch.randn(4 * d, device="cuda", generator=g) * 0.1
    elif kind == "dense":
        st["gu"] = _weight(g, case["bits"], 2 * case["I"], case["H"], case["G"])
        st["dn"] = _weight(g, case["bits"], case["H"], case["I"], case["G"])
        st["x"] = _x(g, case["M"], case["H"])
    else:
        st["layer"] = _layer(g, case["shape"])
        st["x"] = _x(g, case["M"], st["layer"].H, torch.float32)
    return st


# ---- one pass ----------------------------------------------------------------------------------------------------
def _run_f32(st):
    L, x = st["layer"], st["x"]
    M, E, stacked = x.shape[0], L.E, L.shared_stacked
    logits = moe.linear_bf16w(x, L.router)
    ids, coef, err = moe.moe_router(logits, E, L.k, shared_logit=logits[:, E:] if stacked else None, shared_ld=E + 1,
                                    shared_id=E)
    Es = E + (1 if stacked else 0)
    ws, _ = moe.moe_group_routes(ids, Es)
    h = moe.experts_gather_grouped_swiglu(x, L.gate_up, Es, ws, M, L.A)
    shared = None
    if not stacked:
        sh = moe.swiglu(moe.linear_q8(x, L.shared_gate_up, torch.float32), L.I)
        shared = {"s": moe.linear_q8(sh, L.shared_down, torch.float32), "gate_logit": logits[:, E:], "gate_ld": E + 1,
                  "gate_index": E, "err": err}
    y = moe.experts_combine_grouped(h, L.down, Es, ids, coef, ws, M, L.A, shared=shared)
    return {"ids": ids, "coef": coef, "h": h, "y": y}


def run(state):
    kind = state["case"]["kind"]
    if kind == "stack":
        state["graph"].replay()
        return state["out"]
    if kind == "layer":
        return state["layer"].forward(state["x"], ws=state["ws"], out=state["out"], ctx=state["ctx"])
    if kind == "mix":
        h, w_in, inv = moe.hc_mix_down(state["x"], state["down"], state["case"]["r"], True, 1e-6)
        u = moe.hc_mix_up(h, state["up"], state["x"], state["norm"], inv)
        return {"h": h, "w_in": w_in, "inv": inv, "u": u}
    if kind == "dense":
        lin = moe.linear_q8 if state["gu"].bits == 8 else moe.linear_q4
        gu = lin(state["x"], state["gu"])
        h = moe.swiglu(gu, state["dn"].K)
        return {"gu": gu, "h": h, "y": lin(h, state["dn"])}
    return _run_f32(state)


# ---- work and tolerance --------------------------------------------------------------------------------------------
def _qbytes(bits, N, K, G):
    return N * K * bits // 8 + 4 * N * (K // G)


def _touched(c, M, zipf):
    """Experts that M tokens' routes reach: counted on logits of the router's distribution."""
    rng = np.random.default_rng(0)
    bias = -1.1 * zipf * np.log(rng.permutation(c["E"]) + 1.0)
    lg = rng.standard_normal((M, c["E"])) * (0.02 * math.sqrt(c["H"])) + bias
    return len(np.unique(np.argpartition(-lg, c["k"], axis=1)[:, :c["k"]]))


def _layer_work(shape, M, zipf, act_bytes):
    c = SHAPES[shape]
    H, E, I, k = c["H"], c["E"], c["I"], c["k"]
    rows = E + (0 if c["shared"] == "none" else 1)
    expert = _qbytes(c["bits"], 2 * I, H, c["G"]) + _qbytes(c["bits"], H, I, c["G"])
    b = _touched(c, M, zipf) * expert + rows * H * 2 + M * H * act_bytes * 2 + 8 * M * k
    if c["shared"] == "stacked":
        b += expert
    elif c["shared"] == "separate":
        b += _qbytes(8, 2 * I, H, 64) + _qbytes(8, H, I, 64)
    slots = M * (k + (0 if c["shared"] == "none" else 1))
    return b, slots * 6 * H * I + 2 * M * rows * H


def work(case):
    kind = case["kind"]
    if kind == "stack":
        b, f = _layer_work(case["shape"], case["M"], 0.0, 3)
        return {"bytes": LAYERS * b, "flops": LAYERS * f}
    if kind == "layer":
        b, f = _layer_work(case["shape"], case["M"], case["zipf"], 3)
        return {"bytes": b, "flops": f}
    if kind == "mix":
        T, d, r, es = case["T"], case["d"], case["r"], 2 if case["act"] == "bf16" else 4
        b = _qbytes(case["bits"], r + 4, 4 * d, case["G"]) + _qbytes(case["bits"], 4 * d, r, case["G"]) + 16 * d
        return {"bytes": b + T * 5 * d * es + 4 * T * (r + 8), "flops": 2 * T * 4 * d * (2 * r + 4)}
    if kind == "dense":
        M, H, I = case["M"], case["H"], case["I"]
        b = _qbytes(case["bits"], 2 * I, H, case["G"]) + _qbytes(case["bits"], H, I, case["G"])
        return {"bytes": b + 2 * M * (2 * H + 3 * I), "flops": 6 * M * H * I}
    b, f = _layer_work(case["shape"], case["M"], 0.0, 4)
    c = SHAPES[case["shape"]]
    return {"bytes": b + 4 * case["M"] * c["k"] * c["I"], "flops": f}


def tolerance(case):
    # BF16 outputs: one rounding of each result (2^-9 at most, 1.7e-3 in the 2-norm between two that round apart) on top
    # of the intermediate roundings (h, the shared expert's h and s); F16 math adds its operands' roundings
    if case["kind"] in ("stack", "layer", "dense"):
        return {"rel": 1e-2, "max": 0.1}
    if case["kind"] == "mix":
        return {"rel": 8e-3, "max": 4e-2} if case["act"] == "bf16" else {"rel": 1e-5, "max": 1e-3}
    return {"rel": 1e-5, "max": 1e-3}


# ---- 64-bit results --------------------------------------------------------------------------------------------------
def _codes(w, lo, hi, K):
    q = w.q.view(w.N, -1)[lo:hi]
    if w.bits == 8:
        return q.double()
    return torch.stack((q & 15, q >> 4), dim=2).view(hi - lo, K).double()


def _deq(w, lo, hi):
    """Rows lo .. hi of a row-major weight in 64 bits."""
    s = w.scale.view(torch.bfloat16).view(w.N, -1)[lo:hi].double().repeat_interleave(w.G, dim=1)
    m = w.minv.view(torch.bfloat16).view(w.N, -1)[lo:hi].double().repeat_interleave(w.G, dim=1)
    return _codes(w, lo, hi, w.K) * s + m


def _deq_chunk_major(w):
    cb = 32 * w.bits // 8
    q = w.q.view(w.K // 32, w.N, cb).transpose(0, 1).reshape(w.N, -1)
    s = w.scale.view(w.K // w.G, w.N).t().reshape(-1).contiguous()
    m = w.minv.view(w.K // w.G, w.N).t().reshape(-1).contiguous()
    return _deq(moe.QWeight(w.bits, q.reshape(-1).contiguous(), s, m, w.N, w.K, w.G), 0, w.N)


def _silu(v):
    return v * torch.sigmoid(v)


def _exact_layer(L, x):
    """(coef, h by slot, y) of the sublayer."""
    x, E, I, H = x.double(), L.E, L.I, L.H
    logits = x @ L.router.double().t()
    lg = logits[:, :E] + (0.0 if L.router_bias is None else L.router_bias.double())
    top, ids = torch.topk(lg, L.k, dim=1)
    coef = torch.softmax(top, dim=1)
    if L.shared_stacked:
        ids = torch.cat((ids, torch.full_like(ids[:, :1], E)), dim=1)
        coef = torch.cat((coef, torch.sigmoid(logits[:, E:])), dim=1)
    y = torch.zeros((x.shape[0], H), dtype=torch.float64, device="cuda")
    hs = torch.zeros((x.shape[0], L.A, I), dtype=torch.float64, device="cuda")
    for e in torch.unique(ids).tolist():
        m, a = torch.nonzero(ids == e, as_tuple=True)
        gu = x[m] @ _deq(L.gate_up, e * 2 * I, (e + 1) * 2 * I).t()
        hs[m, a] = _silu(gu[:, :I]) * gu[:, I:]
        y.index_add_(0, m, coef[m, a, None] * (hs[m, a] @ _deq(L.down, e * H, (e + 1) * H).t()))
    if L.shared_gate_up is not None:
        gu = x @ _deq(L.shared_gate_up, 0, 2 * I).t()
        s = (_silu(gu[:, :I]) * gu[:, I:]) @ _deq(L.shared_down, 0, H).t()
        y += torch.sigmoid(logits[:, E:]) * s
    return coef, hs.view(-1, I), y


def exact(case, seed):
    kind = case["kind"]
    st = prepare(case, seed)
    if kind in ("stack", "layer"):
        res = []
        pairs = zip(st["layers"], st["x"]) if kind == "stack" else [(st["layer"], st["x"])]
        for L, x in pairs:
            coef, _, y = _exact_layer(L, x)
            res.append({"y": y, "x_out": x.double() + y, "ids": None, "coef": coef, "err": None})
        return res if kind == "stack" else res[0]
    if kind == "mix":
        T, d, r = case["T"], case["d"], case["r"]
        x = st["x"].double().view(T, 4, d)
        inv = torch.rsqrt((x * x).mean(dim=2) + 1e-6)
        n = x * inv[:, :, None]
        z = n.reshape(T, 4 * d) @ _deq(st["down"], 0, r + 4).t() / 4.0
        h, w_in = _silu(z[:, :r]), 2.0 * torch.sigmoid(z[:, r:])
        gate = torch.sigmoid(h @ _deq_chunk_major(st["up"]).t()).view(T, 4, d)
        u = (gate * n * (1.0 + st["norm"].double().view(4, d))).sum(dim=1) / 4.0
        return {"h": h, "w_in": w_in, "inv": inv, "u": u}
    if kind == "dense":
        x, I = st["x"].double(), case["I"]
        gu = x @ _deq(st["gu"], 0, 2 * I).t()
        h = _silu(gu[:, :I]) * gu[:, I:]
        return {"gu": gu, "h": h, "y": h @ _deq(st["dn"], 0, case["H"]).t()}
    coef, h, y = _exact_layer(st["layer"], st["x"])
    return {"ids": None, "coef": coef, "h": h, "y": y}
