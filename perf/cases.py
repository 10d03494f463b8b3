"""The work whose speed counts: calls of the MoE feed-forward path as a serving program makes them.

Shapes are the ones of the repository's benchmark (hidden 2048, experts of 512, 256 experts, top-8 and a shared
expert, vocabulary 248,320).  Weights are random K-quant superblocks whose dequantised values have the spread of a
trained model's (about 0.03), activations are RMS-normalised in size, routing is uniform or Zipf(1.1).
"""
import ctypes
import math

import torch

from breadv2_amd import api

H, I, E, K = 2048, 512, 256, 8
VOCAB = 248320
EPS = 1e-6
Q8, Q4, Q6 = api.QTYPE_Q8_0, api.QTYPE_Q4_K, api.QTYPE_Q6_K
BLOCK = {Q4: (256, 144), Q6: (256, 210), Q8: (32, 34)}
STANDARD = (Q4, Q4, Q6, Q4, Q4, Q6)  # gate, up, down; shared gate, up, down
MIXES = {
    "standard": STANDARD,
    "down_q4": (Q4, Q4, Q4, Q4, Q4, Q4),  # every tensor Q4_K
    "down_q4_shared_q6": (Q4, Q4, Q4, Q4, Q4, Q6),  # the shared expert kept at the higher precision
    "all_q6": (Q6, Q6, Q6, Q6, Q6, Q6),  # a six-bit file
}


def listed():
    return [
        # one expert projection at the reference's fp16 interface: the smallest call, launch latency counts
        {"name": "matvec_512x2048_q4k", "kind": "matvec", "qtype": Q4, "rows": 512, "cols": 2048},
        # one token's logits: the largest single read
        {"name": "lm_head_q6k", "kind": "matvec", "qtype": Q6, "rows": VOCAB, "cols": 2048},
        # the MoE block of one decode token on the fp16 residual stream, norm included
        {"name": "decode_layer_f16", "kind": "f16", "tokens": 1, "routing": "uniform"},
        # one decode token through the whole model's MoE layers
        {"name": "decode_stack_40", "kind": "stack", "tokens": 1, "layers": 40},
        # one token's routed experts with the caller's own routing
        {"name": "expert_block_1", "kind": "block", "tokens": 1, "mix": "standard"},
        # a speculative round: last token and 8 drafts through a run of layers
        {"name": "verify_9x8", "kind": "stack", "tokens": 9, "layers": 8},
        # that round's greedy predictions
        {"name": "greedy_head_9", "kind": "head", "tokens": 9, "qtype": Q4},
        # batched decode, few requests
        {"name": "batch_8_zipf", "kind": "forward", "tokens": 8, "routing": "zipf", "mix": "standard"},
        # batched decode, many requests
        {"name": "batch_64_zipf", "kind": "forward", "tokens": 64, "routing": "zipf", "mix": "standard"},
        # a layer whose file keeps the down projections as Q4_K, an odd number of tokens
        {"name": "batch_27_down_q4", "kind": "forward", "tokens": 27, "routing": "uniform", "mix": "down_q4"},
        # a prefill chunk
        {"name": "prefill_512", "kind": "forward", "tokens": 512, "routing": "uniform", "mix": "standard"},
        # a long prefill chunk
        {"name": "prefill_2048", "kind": "forward", "tokens": 2048, "routing": "uniform", "mix": "standard"},
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["matvec", "matvec", "f16", "stack", "block", "head", "batch", "batch", "mix", "prefill", "prefill"])
    if kind == "matvec":
        qtype = rng.choice([Q4, Q6, Q8])
        cols = 256 * rng.choice([1, 2, 3, 4, 7, 8, 8, 16])
        return {"kind": "matvec", "qtype": qtype, "rows": _log(rng, 200, VOCAB * 2048 // max(cols, 2048)), "cols": cols}
    if kind == "f16":
        return {"kind": "f16", "tokens": _log(rng, 1, 200), "routing": rng.choice(["uniform", "zipf"])}
    if kind == "stack":
        tokens = rng.choice([1, 1, _log(rng, 2, 20)])
        return {"kind": "stack", "tokens": tokens, "layers": rng.randint(2, 40 if tokens == 1 else 8)}
    if kind == "block":
        return {"kind": "block", "tokens": _log(rng, 1, 12), "mix": rng.choice(sorted(MIXES))}
    if kind == "head":
        return {"kind": "head", "tokens": _log(rng, 1, 32), "qtype": rng.choice([Q4, Q4, Q6])}
    if kind == "batch":
        return {"kind": "forward", "tokens": _log(rng, 2, 130), "routing": rng.choice(["uniform", "zipf"]), "mix": "standard"}
    if kind == "mix":
        return {"kind": "forward", "tokens": _log(rng, 1, 130), "routing": rng.choice(["uniform", "zipf"]),
                "mix": rng.choice([m for m in sorted(MIXES) if m != "standard"])}
    return {"kind": "forward", "tokens": _log(rng, 130, 2048), "routing": rng.choice(["uniform", "zipf"]), "mix": "standard"}


# ------------------------------------------------------------------ inputs


def _bytes(n, gen):
    words = torch.empty((n + 3) // 4, dtype=torch.int32, device="cuda")
    words.random_(-(2**31), 2**31, generator=gen)
    return words.view(torch.uint8)[:n]


def _fp16_scale(n, mean, gen):
    u = torch.rand(n, device="cuda", generator=gen)
    return (mean * (0.5 + u)).half().view(torch.uint8).view(n, 2)


def _quant(qtype, elems, gen):
    """Random superblocks of `elems` weights as bytes; dequantised values of about 0.03 around zero."""
    per, size = BLOCK[qtype]
    n = elems // per
    b = _bytes(n * size, gen).view(n, size)
    if qtype == Q4:  # d, dmin, 12 scale bytes, 128 nibble pairs
        b[:, 0:2] = _fp16_scale(n, 1.5e-4, gen)
        b[:, 2:4] = _fp16_scale(n, 1.1e-3, gen)
    elif qtype == Q6:  # ql, qh, 16 int8 scales, d
        b[:, 208:210] = _fp16_scale(n, 2.2e-5, gen)
    else:  # d, 32 int8
        b[:, 0:2] = _fp16_scale(n, 4e-4, gen)
    return b.view(-1)


def _gen(seed, part=0):
    g = torch.Generator(device="cuda")
    g.manual_seed(1000003 * int(seed) + 7919 * part + 1)
    return g


def _layer(mix, gen, zipf):
    """One layer's tensors: six quantised ones, router, shared gate, post-attention norm."""
    t = MIXES[mix]
    n = I * H
    q = [_quant(t[0], E * n, gen), _quant(t[1], E * n, gen), _quant(t[2], E * n, gen),
         _quant(t[3], n, gen), _quant(t[4], n, gen), _quant(t[5], n, gen)]
    router = 0.02 * torch.randn(E, H, device="cuda", generator=gen)
    if zipf:  # the last activation feature is 1: its column is the routing bias
        p = torch.arange(1, E + 1, device="cuda", dtype=torch.float64) ** -1.1
        order = torch.randperm(E, device="cuda", generator=gen)
        router[order, H - 1] = torch.log(p / p.sum()).float()
    shgate = (0.02 * torch.randn(H, device="cuda", generator=gen)).half()
    norm = 1.0 + 0.1 * torch.randn(H, device="cuda", generator=gen)
    tensors = api.LayerTensors(api.shape(H, I, I, E, K, EPS), *q, router, shgate, t)
    return tensors, norm


def _inputs(case, seed):
    """The tensors of a case, from the seed alone."""
    g, kind = _gen(seed), case["kind"]
    if kind == "matvec":
        w = _quant(case["qtype"], case["rows"] * case["cols"], g)
        return {"w": w, "x": torch.randn(case["cols"], device="cuda", generator=g).half()}
    if kind == "head":
        w = _quant(case["qtype"], VOCAB * H, g)
        return {"w": w, "hidden": 4.0 * torch.randn(case["tokens"], H, device="cuda", generator=g),
                "norm": 1.0 + 0.1 * torch.randn(H, device="cuda", generator=g)}
    n = case["tokens"]
    d = {"layers": [_layer(case.get("mix", "standard"), _gen(seed, 1 + l), case.get("routing") == "zipf")
                    for l in range(case.get("layers", 1))]}
    x = torch.randn(n, H, device="cuda", generator=g)
    if kind == "f16":
        d["hidden"] = (2.0 * x).half()
        if case["routing"] == "zipf":  # feature H - 1 of the normalised activations is close to 1
            d["hidden"][:, H - 1] = 2.0
    elif kind == "stack":
        d["hidden"] = 2.0 * x
    else:
        if case.get("routing") == "zipf":
            x[:, H - 1] = 1.0
        d["x"] = x
        d["hidden"] = 2.0 * torch.randn(n, H, device="cuda", generator=g)
    if kind == "block":
        d["idx"] = torch.stack([torch.randperm(E, device="cuda", generator=g)[:K] for _ in range(n)]).int()
        w = torch.rand(n, K, device="cuda", generator=g) + 0.05
        d["w_routed"] = w / w.sum(1, keepdim=True)
    return d


def prepare(case, seed):
    d = _inputs(case, seed)
    kind = case["kind"]
    if kind == "matvec":
        d["y"] = torch.empty(case["rows"], dtype=torch.float16, device="cuda")
    else:
        d["ctx"] = api.MoeContext(api.shape(H, I, I, E, K, EPS), max_tokens=case["tokens"])
    if "layers" in d:
        d["desc"] = []
        for t, norm in d["layers"]:
            m = t.desc()
            m.post_norm_w = ctypes.c_void_p(norm.data_ptr())
            d["desc"].append(m)
    if kind == "f16":
        d["normed"] = torch.empty_like(d["hidden"])
    d["case"] = dict(case)
    return d


# ------------------------------------------------------------------ one pass


def run(state):
    c, kind = state["case"], state["case"]["kind"]
    if kind == "matvec":
        api.bread_matvec(state["w"], state["x"], state["y"], c["rows"], c["cols"], c["qtype"])
        return state["y"]
    ctx, n = state["ctx"], c["tokens"]
    if kind == "head":
        tokens, logits = ctx.greedy_head(state["hidden"], state["norm"], state["w"], c["qtype"], VOCAB, n)
        return {"logits": logits, "tokens": tokens}
    if kind == "f16":
        ctx.forward_f16(state["desc"][0], state["hidden"], state["normed"], n, norm_w=state["layers"][0][1])
        return {"hidden": state["hidden"], "normed": state["normed"]}
    if kind == "stack":
        if n == 1:
            ctx.decode_layers(state["desc"], state["hidden"])
        else:
            ctx.stack_forward(state["desc"], state["hidden"], n)
    elif kind == "block":
        ctx.expert_block(state["desc"][0], state["x"], state["hidden"], n, state["idx"], state["w_routed"])
    else:
        ctx.forward(state["desc"][0], state["x"], state["hidden"], n)
    return state["hidden"]


# ------------------------------------------------------------------ what a pass cannot do without


def _row(qtype, cols):
    per, size = BLOCK[qtype]
    return cols // per * size


def _distinct(tokens, routing):
    """Experts that at least one of the tokens chooses, expected."""
    if routing != "zipf":
        return E * (1.0 - (1.0 - K / E) ** tokens)
    # a token takes expert r when log p_r plus its own logit, N(0, 0.02^2 H), is above a bar; K do on average
    spread = 0.02 * math.sqrt(H)
    bias = [-1.1 * math.log(r + 1) for r in range(E)]

    def takes(bar):
        return [0.5 * math.erfc((bar - b) / (spread * math.sqrt(2.0))) for b in bias]

    lo, hi = -20.0, 20.0
    for _ in range(60):
        bar = 0.5 * (lo + hi)
        lo, hi = (bar, hi) if sum(takes(bar)) > K else (lo, bar)
    return sum(1.0 - (1.0 - q) ** tokens for q in takes(lo))


def work(case):
    kind = case["kind"]
    if kind == "matvec":
        r, c = case["rows"], case["cols"]
        return {"bytes": r * _row(case["qtype"], c) + 2 * c + 2 * r, "flops": 2 * r * c}
    n = case["tokens"]
    if kind == "head":
        return {"bytes": VOCAB * _row(case["qtype"], H) + n * (4 * H + 2 * VOCAB + 4) + 4 * H, "flops": 2 * n * VOCAB * H}
    t = MIXES[case.get("mix", "standard")]
    expert = I * (_row(t[0], H) + _row(t[1], H)) + H * _row(t[2], I)
    shared = I * (_row(t[3], H) + _row(t[4], H)) + H * _row(t[5], I)
    if kind == "block":
        d = _distinct(n, "uniform")
        return {"bytes": d * expert + n * (12 * H + 8 * K), "flops": 6 * n * K * I * H}
    d = _distinct(n, case.get("routing"))
    io = {"f16": 6 * H + 4 * H / n, "stack": 4 * H / n, "forward": 12 * H}[kind]
    per_layer = d * expert + shared + 4 * E * H + 2 * H
    layers = case.get("layers", 1)
    return {"bytes": layers * (per_layer + n * io) + (8 * H * n if kind == "stack" else 0),
            "flops": layers * n * (6 * (K + 1) * I * H + 2 * E * H + 2 * H)}


def tolerance(case):
    """About four times the largest error against 64 bits that the path shows at each precision."""
    kind = case["kind"]
    if kind in ("matvec", "head", "f16"):
        return {"rel": 1e-3, "max": 4e-3}  # rounding to fp16 alone: 2.1e-4
    if kind == "block" or case.get("mix", "standard") != "standard":
        return {"rel": 4e-6, "max": 1e-4}  # fp32 sums of 2048 and 512 products: 6e-7
    if kind == "stack":  # each layer's error travels on through the ones behind it: 1.6e-4 over 40 layers
        return {"rel": 8e-4, "max": 4e-2} if case["tokens"] <= 16 else {"rel": 2e-3, "max": 8e-2}
    if case["tokens"] <= 16:
        return {"rel": 1e-4, "max": 2e-3}  # gate and up on 16-bit fixed-point activations: 2.2e-5
    return {"rel": 1e-3, "max": 1e-2}  # weights rounded to fp16: 2.5e-4


# ------------------------------------------------------------------ in 64 bits, in plain torch


def _f16(b, at):
    return b[:, at:at + 2].contiguous().view(torch.float16).double()


def _dequant(w, qtype, rows, cols):
    per, size = BLOCK[qtype]
    b = w.view(-1, size)
    n = b.shape[0]
    if qtype == Q8:
        v = _f16(b, 0) * b[:, 2:].contiguous().view(torch.int8).double()
    elif qtype == Q4:
        s = b[:, 4:16].int()
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double()
        m = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        q = b[:, 16:].view(n, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).view(n, 8, 32).double()
        v = (_f16(b, 0) * sc)[:, :, None] * q - (_f16(b, 2) * m)[:, :, None]
    else:
        ql, qh = b[:, 0:128].view(n, 2, 64).int(), b[:, 128:192].view(n, 2, 32).int()
        lo, hi = ql & 15, ql >> 4
        parts = [lo[:, :, :32] | ((qh & 3) << 4), lo[:, :, 32:] | (((qh >> 2) & 3) << 4),
                 hi[:, :, :32] | (((qh >> 4) & 3) << 4), hi[:, :, 32:] | ((qh >> 6) << 4)]
        q = torch.stack(parts, 2).view(n, 16, 16).double() - 32.0
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        v = (_f16(b, 208) * sc)[:, :, None] * q
    return v.reshape(rows, cols)


def _expert(t, types, which, e, x):
    """down(silu(gate x) * up x) for the rows of x; e is None for the shared expert."""
    g, u, d = (t.gate_exps, t.up_exps, t.down_exps) if which == 0 else (t.gate_sh, t.up_sh, t.down_sh)
    tg, tu, td = types[3 * which:3 * which + 3]
    if e is not None:
        g, u, d = (w.view(E, -1)[e] for w in (g, u, d))
    a = x @ _dequant(g, tg, I, H).T
    a = a * torch.sigmoid(a) * (x @ _dequant(u, tu, I, H).T)
    return a @ _dequant(d, td, H, I).T


def _moe(t, types, x, idx=None, w=None):
    out = torch.zeros_like(x)
    if idx is None:
        p = torch.softmax(x @ t.router.double().T, 1)
        w, idx = torch.topk(p, K, dim=1)
        w = w / w.sum(1, keepdim=True)
        out += torch.sigmoid(x @ t.shgate.double())[:, None] * _expert(t, types, 1, None, x)
    for e in torch.unique(idx).tolist():
        rows, rank = torch.nonzero(idx == e, as_tuple=True)
        out.index_add_(0, rows, w[rows, rank][:, None] * _expert(t, types, 0, e, x[rows]))
    return out


def _rms(h, norm):
    return h / torch.sqrt((h * h).mean(1, keepdim=True) + EPS) * norm.double()


def exact(case, seed):
    d = _inputs(case, seed)
    kind = case["kind"]
    if kind == "matvec":
        rows, cols, x = case["rows"], case["cols"], d["x"].double()
        w = d["w"].view(rows, -1)
        return torch.cat([_dequant(p.reshape(-1), case["qtype"], p.shape[0], cols) @ x for p in w.split(16384)])
    if kind == "head":
        x = _rms(d["hidden"].double(), d["norm"]).half().double()
        w = d["w"].view(VOCAB, -1)
        y = [x @ _dequant(p.reshape(-1), case["qtype"], p.shape[0], H).T for p in w.split(16384)]
        return {"logits": torch.cat(y, 1), "tokens": None}
    types, h = MIXES[case.get("mix", "standard")], d["hidden"].double()
    if kind == "f16":
        x = _rms(h, d["layers"][0][1]).half().double()
        return {"hidden": h + _moe(d["layers"][0][0], types, x), "normed": x}
    if kind == "stack":
        for t, norm in d["layers"]:
            h = h + _moe(t, types, _rms(h, norm))
        return h
    if kind == "block":
        return h + _moe(d["layers"][0][0], types, d["x"].double(), d["idx"].long(), d["w_routed"].double())
    return h + _moe(d["layers"][0][0], types, d["x"].double())
