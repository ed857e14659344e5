"""The work this library is used for, as cases to time and compare.

A case is one call of a public entry point on the shapes that the benchmark,
the tests and the model configurations of this repository use: the MoE layer
(nx_moe_forward_dev), the whole MoE block with its norm and router
(nx_moe_block_dev) and the dense projections (nx_matvec_dev), from one token
(a decode step) over decode batches to prefill.  Token counts of batches are
odd on purpose: a serving batch is whatever is running.

Weights are drawn from N(0, 0.02) and quantized here, in plain torch, to the
GGUF block layouts, so that exact() can evaluate the same payload in 64 bits
without the library.
"""
import math

import torch

import nexus_amd as nx

FORMATS = {"Q4_K": nx.Q4_K, "Q8_0": nx.Q8_0, "Q4_0": nx.Q4_0}
BLOCK = {"Q4_K": (256, 144), "Q8_0": (32, 34), "Q4_0": (32, 18)}
EPS = 1e-5

# expert-layer shapes of the repository's model configurations
MODELS = {
    "mixtral": dict(experts=8, hidden=4096, ffn=14336, top_k=2, shared_ffn=0, sigmoid=False),
    "qwen3": dict(experts=128, hidden=2048, ffn=768, top_k=8, shared_ffn=0, sigmoid=False),
    "deepseek": dict(experts=256, hidden=7168, ffn=2048, top_k=8, shared_ffn=2048, sigmoid=True),
}
# dense projections of a decoder layer and the output head: (rows, cols)
PROJECTIONS = {"attn_q": (4096, 4096), "attn_k": (1024, 4096), "qwen3_q": (4096, 2048),
               "deepseek_o": (7168, 2048)}
HEAD = (32000, 4096)


def _moe(kind, model, fmt, tokens, skew=0.0):
    return dict(MODELS[model], kind=kind, fmt=fmt, tokens=tokens, skew=skew)


def _matvec(fmt, rows, cols, tokens):
    return dict(kind="matvec", fmt=fmt, rows=rows, cols=cols, tokens=tokens)


def listed():
    cases = {
        # one decode step of one sequence: the whole FFN half of a layer, with
        # routing bit-identical to the reference; latency
        "block_mixtral_q4k_1": _moe("block", "mixtral", "Q4_K", 1),
        # the same through the layer alone, on many small experts
        "moe_qwen3_q4k_1": _moe("forward", "qwen3", "Q4_K", 1),
        # a handful of sequences decoding together
        "moe_mixtral_q4_0_7": _moe("forward", "mixtral", "Q4_0", 7),
        # decode batches of a server: few tokens per expert
        "moe_mixtral_q4k_32": _moe("forward", "mixtral", "Q4_K", 32),
        "moe_qwen3_q4k_61": _moe("forward", "qwen3", "Q4_K", 61),
        # the largest weights, with sigmoid scores and a shared expert
        "moe_deepseek_q4k_27": _moe("forward", "deepseek", "Q4_K", 27),
        # prefill of a short prompt: tens of tokens per expert
        "moe_qwen3_q4k_509": _moe("forward", "qwen3", "Q4_K", 509),
        # prefill with unevenly used experts
        "moe_mixtral_q8_0_2048": _moe("forward", "mixtral", "Q8_0", 2048, skew=1.2),
        # prefill of a long prompt through a whole block (the largest case)
        "block_deepseek_q4k_4096": _moe("block", "deepseek", "Q4_K", 4096),
        # a projection of one decode step (the smallest call)
        "proj_q4k_1": _matvec("Q4_K", 4096, 4096, 1),
        # the output head of a decode batch
        "head_q8_0_13": _matvec("Q8_0", 32000, 4096, 13),
        # a projection over a prompt
        "proj_q4k_509": _matvec("Q4_K", 4096, 4096, 509),
    }
    return [dict(c, name=n) for n, c in cases.items()]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    fmt = rng.choice(["Q4_K", "Q4_K", "Q8_0", "Q4_0"])
    kind = rng.choice(["forward", "forward", "block", "matvec"])
    if kind == "matvec":
        if rng.random() < 0.25:
            return _matvec(fmt, *HEAD, _log_int(rng, 1, 32))
        return _matvec(fmt, *PROJECTIONS[rng.choice(sorted(PROJECTIONS))], _log_int(rng, 1, 1024))
    model = rng.choice(sorted(MODELS))
    # prefills of the large models stay below the largest listed case
    case = _moe(kind, model, fmt, _log_int(rng, 1, 2048), rng.choice([0.0, 0.0, 1.2]))
    if model != "deepseek" and rng.random() < 0.3:  # other expert widths
        case["ffn"] = 256 * _log_int(rng, 2, 28)
    return case


# ---------------------------------------------------------------- weights
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(1000003 * seed + 17)
    return g


def _bytes_of_half(v):
    return v.to(torch.float16).view(torch.uint8).reshape(v.shape[0], 2)


def _quantize(fmt, w):
    """The GGUF payload of the float weights w (their count a whole number of blocks)."""
    b = w.reshape(-1, BLOCK[fmt][0])
    if fmt == "Q8_0":
        d = b.abs().amax(1) / 127.0
        q = torch.round(b / d[:, None]).to(torch.int8).view(torch.uint8)
        return torch.cat([_bytes_of_half(d), q], 1).reshape(-1)
    if fmt == "Q4_0":
        d = b.abs().amax(1) / 7.0
        q = (torch.round(b / d[:, None]) + 8).to(torch.uint8)
        return torch.cat([_bytes_of_half(d), q[:, :16] | (q[:, 16:] << 4)], 1).reshape(-1)
    sub = b.reshape(-1, 8, 32)
    low = (-sub.amin(2)).clamp_(min=0)
    scale = (sub.amax(2) + low) / 15.0
    d, dmin = scale.amax(1) / 63.0, low.amax(1) / 63.0
    sc, mn = torch.round(scale / d[:, None]), torch.round(low / dmin[:, None])
    q = torch.round((sub + (dmin[:, None] * mn)[:, :, None]) / (d[:, None] * sc)[:, :, None])
    q = q.clamp_(0, 15).to(torch.uint8).reshape(-1, 256)
    sc, mn = sc.to(torch.uint8), mn.to(torch.uint8)
    packed = torch.cat([sc[:, :4] | ((sc[:, 4:] >> 4) << 6), mn[:, :4] | ((mn[:, 4:] >> 4) << 6),
                        (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)], 1)
    return torch.cat([_bytes_of_half(d), _bytes_of_half(dmin), packed,
                      q[:, :128] | (q[:, 128:] << 4)], 1).reshape(-1)


def _half_at(p, at):
    return p[:, at:at + 2].contiguous().view(torch.float16).to(torch.float64)


def _dequantize(fmt, payload, rows, cols):
    """The weights of a payload in 64 bits, as GGUF defines them."""
    p = payload.reshape(-1, BLOCK[fmt][1])
    d = _half_at(p, 0)
    if fmt == "Q8_0":
        w = d * p[:, 2:].contiguous().view(torch.int8)
    elif fmt == "Q4_0":
        w = d * (torch.cat([p[:, 2:] & 15, p[:, 2:] >> 4], 1).to(torch.float64) - 8)
    else:
        a, b, c = p[:, 4:8], p[:, 8:12], p[:, 12:16]
        sc = torch.cat([a & 63, (c & 15) | ((a >> 6) << 4)], 1)
        mn = torch.cat([b & 63, (c >> 4) | ((b >> 6) << 4)], 1)
        q = torch.cat([p[:, 16:] & 15, p[:, 16:] >> 4], 1).reshape(-1, 8, 32)
        w = (d * sc)[:, :, None] * q - (_half_at(p, 2) * mn)[:, :, None]
    return w.reshape(rows, cols)


def _roles(case, width):
    H = case["hidden"]
    return ((nx.ROLE_GATE, width, H), (nx.ROLE_UP, width, H), (nx.ROLE_DOWN, H, width))


def _members(case):
    yield from ((e, case["ffn"]) for e in range(case["experts"]))
    if case["shared_ffn"]:
        yield nx.EXPERT_SHARED, case["shared_ffn"]


def _payload(case, seed, index, rows, cols):
    g = _generator(seed * 4096 + index)
    return _quantize(case["fmt"], torch.randn((rows, cols), generator=g, device="cuda") * 0.02)


def _inputs(case, seed):
    """x (or the hidden state), and what the case's router needs."""
    g = _generator(seed * 4096 + 4095)
    if case["kind"] == "matvec":
        return {"x": torch.randn((case["tokens"], case["cols"]), generator=g, device="cuda")}
    T, H, E = case["tokens"], case["hidden"], case["experts"]
    got = {"x": torch.randn((T, H), generator=g, device="cuda"),
           "router": torch.randn((E, H), generator=g, device="cuda") * 0.02}
    if case["kind"] == "block":
        got["norm"] = 1.0 + 0.1 * torch.randn((H,), generator=g, device="cuda")
    else:
        popularity = -case["skew"] * torch.log(torch.arange(1, E + 1, device="cuda"))
        got["logits"] = (got["x"] @ got["router"].t() + popularity).contiguous()
    return got


# ---------------------------------------------------------------- the call
_shared = {}


def _context():
    """One context on one stream that torch uses too, as a program keeps it."""
    if not _shared:
        stream = torch.cuda.Stream()
        torch.cuda.set_stream(stream)
        ctx = nx.Context(0)
        ctx.set_stream(stream.cuda_stream)
        _shared.update(ctx=ctx, stream=stream)
    return _shared["ctx"]


def prepare(case, seed):
    ctx = _context()
    fmt = FORMATS[case["fmt"]]
    state = dict(_inputs(case, seed), case=case)
    if case["kind"] == "matvec":
        rows, cols = case["rows"], case["cols"]
        payload = _payload(case, seed, 0, rows, cols)
        state["weights"] = nx.Matrix(ctx, fmt, rows, cols)
        state["weights"].load_dev(payload.data_ptr(), payload.numel())
        state["out"] = torch.empty((case["tokens"], rows), device="cuda")
        return state
    ex = nx.Experts(ctx, fmt, case["experts"], case["hidden"], case["ffn"],
                    shared_ff_dim=case["shared_ffn"])
    for i, (e, width) in enumerate(_members(case)):
        for role, rows, cols in _roles(case, width):
            payload = _payload(case, seed, 3 * i + role, rows, cols)
            ex.load_dev(e, role, payload.data_ptr(), payload.numel())
    state["weights"] = ex
    state["out"] = torch.empty_like(state["x"])
    return state


def run(state):
    case, w, x, out = state["case"], state["weights"], state["x"], state["out"]
    T = case["tokens"]
    if case["kind"] == "matvec":
        w.matvec_dev(x.data_ptr(), x.numel(), T, out.data_ptr())
        return out
    mode = nx.SCORE_SIGMOID if case["sigmoid"] else nx.SCORE_SOFTMAX
    if case["kind"] == "block":
        # the block updates the hidden state in place
        out.copy_(x)
        w.block_dev(out.data_ptr(), state["norm"].data_ptr(), state["norm"].numel(), EPS,
                    state["router"].data_ptr(), state["router"].numel(), T, case["top_k"], mode)
    else:
        w.forward_dev(x.data_ptr(), state["logits"].data_ptr(), T, case["top_k"],
                      out.data_ptr(), mode)
    return out


# ---------------------------------------------------------------- what it takes
def _per_weight(case):
    return BLOCK[case["fmt"]][1] / BLOCK[case["fmt"]][0]


def work(case):
    T = case["tokens"]
    if case["kind"] == "matvec":
        n = case["rows"] * case["cols"]
        return {"bytes": n * _per_weight(case) + 4 * T * (case["rows"] + case["cols"]),
                "flops": 2 * n * T}
    E, H, k = case["experts"], case["hidden"], case["top_k"]
    active = E * (1.0 - (1.0 - k / E) ** T)
    weights = 3 * H * (active * case["ffn"] + case["shared_ffn"])
    flops = 6 * T * H * (k * case["ffn"] + case["shared_ffn"])
    moved = weights * _per_weight(case) + 8 * T * H
    if case["kind"] == "block":
        moved += 4 * E * H + 4 * H
        flops += 2 * T * E * H
    else:
        moved += 4 * T * E
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    """Dense products and decode batches sum in 32 bits; from about three
    tokens per expert (or a shared expert and a few tokens) the layer may take
    the grouped GEMM, whose operands and per-route rows are bf16 (4.4e-3 from
    exact()).  Below that, four times what was measured against exact():
    Q4_K 1.5e-6, and on the matrix cores Q8_0 4.3e-6 and Q4_0 8.3e-5, whose
    code operands fill fewer bits; dense products 3.1e-7."""
    if case["kind"] == "matvec":
        return {"rel": 2e-6, "max": 2e-5}
    T, E, k = case["tokens"], case["experts"], case["top_k"]
    active = E * (1.0 - (1.0 - k / E) ** T)
    per_expert = T * k / active
    if case["shared_ffn"]:
        bf16 = per_expert >= 8.0 or (case["fmt"] != "Q4_K" and T >= 6)
    else:
        bf16 = per_expert >= 12.0
    if bf16:
        return {"rel": 1.5e-2, "max": 1.5e-1}
    rel = {"Q4_K": 6e-6, "Q8_0": 2e-5, "Q4_0": 4e-4}[case["fmt"]]
    return {"rel": rel, "max": 10 * rel}


# ---------------------------------------------------------------- in 64 bits
def _routes(case, logits):
    """Experts and weights of each token: the top-k logits (ties to the lower
    index), softmax over the selected or sigmoid scores that sum to 1."""
    top, idx = torch.sort(logits, dim=1, descending=True, stable=True)
    top, idx = top[:, :case["top_k"]], idx[:, :case["top_k"]]
    if case["sigmoid"]:
        s = torch.sigmoid(top)
        return idx, s / s.sum(1, keepdim=True)
    return idx, torch.softmax(top, 1)


def exact(case, seed):
    _context()
    got = _inputs(case, seed)
    x = got["x"].double()
    fmt = case["fmt"]
    if case["kind"] == "matvec":
        w = _dequantize(fmt, _payload(case, seed, 0, case["rows"], case["cols"]), case["rows"],
                        case["cols"])
        return x @ w.t()
    out = torch.zeros_like(x)
    if case["kind"] == "block":
        out += x
        x = x / torch.sqrt((x * x).mean(1, keepdim=True) + EPS) * got["norm"].double()
        logits = x @ got["router"].double().t()
    else:
        logits = got["logits"].double()
    idx, weight = _routes(case, logits)
    for i, (e, width) in enumerate(_members(case)):
        if e == nx.EXPERT_SHARED:
            token, share = torch.arange(len(x), device="cuda"), torch.ones(len(x), device="cuda").double()
        else:
            token, slot = torch.nonzero(idx == e, as_tuple=True)
            share = weight[token, slot]
        if not len(token):
            continue
        gate, up, down = (_dequantize(fmt, _payload(case, seed, 3 * i + role, rows, cols), rows, cols)
                          for role, rows, cols in _roles(case, width))
        xe = x[token]
        g = xe @ gate.t()
        y = (g * torch.sigmoid(g) * (xe @ up.t())) @ down.t()
        out.index_add_(0, token, y * share[:, None])
    return out
