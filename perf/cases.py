"""The work a user of this framework has it do, as measurable cases.

Every case goes through the public Python surface: the MoE blocks and the
expert seam of ``pagedmoe_amd.streaming`` (resident and paged) and the format
functions of ``pagedmoe_amd.kernels``.  Shapes are the ones the benchmark and
the tests use:

  tiny  hidden  1024, inter  512,  32 experts, top-4,  4-bit, softmax
  q235  hidden  4096, inter 1536, 128 experts, top-8,  4-bit, softmax
        (Qwen3-235B-shaped)
  next  hidden  2048, inter  512, 512 experts, top-10, 6-bit, softmax, a
        sigmoid-gated shared expert (Qwen3-Next-shaped)
  dsv3  hidden  7168, inter 2048, 384 experts, top-8,  4-bit, sigmoid scores
        in 8 groups of which 4 are kept, scale 2.5, a shared expert
        (DeepSeek-V3-shaped)

A block case of several layers calls each layer's block on hidden states of
its own, as a decode step of a model does, so a layer's experts come from HBM
and not from the last-level cache.  Weights are drawn in the checkpoint's own
format (packed words, bf16 scales and biases), with the bell-shaped codes that
a min/max quantizer gives for normal weights.
"""

from __future__ import annotations

import math

import torch

SHAPES = {
    "tiny": dict(hidden=1024, inter=512, experts=32, k=4, bits=4, scoring="softmax", shared=0),
    "q235": dict(hidden=4096, inter=1536, experts=128, k=8, bits=4, scoring="softmax", shared=0),
    "next": dict(hidden=2048, inter=512, experts=512, k=10, bits=6, scoring="softmax", shared=1),
    "dsv3": dict(hidden=7168, inter=2048, experts=384, k=8, bits=4, scoring="sigmoid", shared=1),
}
N_GROUP, TOPK_GROUP, ROUTED_SCALE = 8, 4, 2.5
PROJS = ("gate_proj", "up_proj", "down_proj")
STD = 0.02  # of weights and router rows


# ---------------------------------------------------------------- the cases

def listed() -> list:
    return [
        # one token of a small model: nothing but latency and launches
        _block("tiny_decode_1", "tiny", 1, layers=1),
        # interactive decode of one sequence, several layers of a token's pass
        _block("q235_decode_1", "q235", 1, layers=4),
        _block("dsv3_decode_1", "dsv3", 1, layers=2),
        # small serving batch
        _block("q235_decode_8", "q235", 8, layers=2),
        # a draft of 8 tokens verified in one call, 6-bit weights
        _block("next_verify_8", "next", 8, layers=2),
        # a serving batch of an odd size
        _block("q235_batch_29", "q235", 29, layers=1),
        # the seam under a caller's own routing: a short prompt or a large
        # batch, per-slot outputs uncombined
        {"name": "q235_seam_100", "kind": "seam", "shape": "q235", "n": 100},
        # prompts in one chunk: a ragged 6-bit one, and 4-bit ones with the
        # uneven expert loads of a trained router
        _block("next_prefill_1000", "next", 1000, layers=1),
        _block("q235_prefill_2048", "q235", 2048, layers=1, skew=True),
        # the largest chunk: a long prompt through the fused prefill pass
        _block("q235_prefill_16384", "q235", 16384, layers=1, skew=True),
        # experts paged between host memory and HBM: a few tokens decoded one
        # after the other through two layers, half of the experts resident
        {"name": "q235_paged_decode", "kind": "paged", "shape": "q235", "n": 8, "layers": 2,
         "slots": 160},
        # making a checkpoint: a stack of gate projections into the packed
        # format and back
        {"name": "format_24576x4096_4bit", "kind": "format", "rows": 24576, "cols": 4096,
         "bits": 4},
    ]


def _block(name, shape, n, layers, skew=False):
    return {"name": name, "kind": "block", "shape": shape, "n": n, "layers": layers, "skew": skew}


# most tokens of a drawn call: no case costs more than the 16384-token one
MOST_TOKENS = {"tiny": 16384, "q235": 16384, "next": 16384, "dsv3": 2048}


def draw(rng) -> dict:
    kind = rng.choices(["block", "seam", "paged", "format"], [12, 3, 1, 2])[0]
    if kind == "format":
        bits = rng.choice([4, 6])
        cols = 64 * _log_int(rng, 8, 128)
        if bits == 6:
            cols = 512 * max(1, cols // 512)
        return {"kind": kind, "rows": _log_int(rng, 512, 32768), "cols": cols, "bits": bits}
    if kind == "paged":
        return {"kind": kind, "shape": rng.choice(["tiny", "q235"]), "n": rng.randint(1, 12),
                "layers": 2, "slots": 0}
    shape = rng.choice(["tiny", "q235", "q235", "next", "dsv3"])
    n = _log_int(rng, 1, MOST_TOKENS[shape])
    if kind == "seam":
        n = min(n, 2048)
        return {"kind": kind, "shape": shape, "n": n}
    return {"kind": kind, "shape": shape, "n": n, "layers": 2 if n <= 8 else 1,
            "skew": n > 64 and rng.random() < 0.5}


def _log_int(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


# ---------------------------------------------------------------- inputs

def _gen(seed: int, *what: int) -> torch.Generator:
    s = seed
    for w in what:
        s = (s * 1000003 + w + 1) % (1 << 62)
    return torch.Generator(device="cuda").manual_seed(s)


def _codes(shape, bits: int, gen) -> torch.Tensor:
    """uint8 quantizer codes with the spread of a quantized normal weight."""
    a = torch.randint(0, 128, shape, dtype=torch.uint8, device="cuda", generator=gen)
    a += torch.randint(0, 128, shape, dtype=torch.uint8, device="cuda", generator=gen)
    return a.bitwise_right_shift_(8 - bits)


def _pack(q: torch.Tensor, bits: int) -> torch.Tensor:
    """Little-endian bit stream per row as int32 words."""
    if bits == 4:
        b = q[..., 0::2] | (q[..., 1::2] << 4)
    else:
        q0, q1, q2, q3 = (q[..., i::4] for i in range(4))
        b = torch.stack((q0 | (q1 << 6), (q1 >> 2) | (q2 << 4), (q2 >> 4) | (q3 << 2)), dim=-1)
    return b.reshape(*q.shape[:-1], -1).contiguous().view(torch.int32)


def _expert_chunks(sh: dict, seed: int, layer: int):
    """(first expert, {projection: (codes, scales, biases)}) for the routed
    experts and, last, the shared one, a few experts at a time."""
    d, i, bits = sh["hidden"], sh["inter"], sh["bits"]
    total = sh["experts"] + sh["shared"]
    per = max(1, (1 << 28) // (d * i))
    top = float((1 << bits) - 1)
    for e0 in range(0, total, per):
        ne = min(per, total - e0)
        gen = _gen(seed, 7, layer, e0)
        part = {}
        for proj in PROJS:
            rows, cols = (d, i) if proj == "down_proj" else (i, d)
            q = _codes((ne, rows, cols), bits, gen)
            r = torch.rand((2, ne, rows, cols // 64), device="cuda", generator=gen)
            s = (4.8 * STD / top * (0.8 + 0.4 * r[0])).to(torch.bfloat16)
            b = (-0.5 * top * s.float() * (0.9 + 0.2 * r[1])).to(torch.bfloat16)
            part[proj] = (q, s, b)
        yield e0, part


def _fill(slab, sh: dict, seed: int, layer: int) -> None:
    for e0, part in _expert_chunks(sh, seed, layer):
        for proj, (q, s, b) in part.items():
            e1 = e0 + q.shape[0]
            slab.compute(proj + ".weight")[e0:e1].copy_(_pack(q, sh["bits"]))
            slab.compute(proj + ".scales")[e0:e1].copy_(s)
            slab.compute(proj + ".biases")[e0:e1].copy_(b)


def _router(case: dict, seed: int, layer: int) -> dict:
    """Router rows, and the bias, skew and shared-gate tensors a shape has."""
    sh = SHAPES[case["shape"]]
    gen = _gen(seed, 3, layer)
    e, d = sh["experts"], sh["hidden"]
    r = {"gate": (torch.randn((e, d), device="cuda", generator=gen) * STD).to(torch.bfloat16)}
    r["bias"] = torch.randn(e, device="cuda", generator=gen) * 0.05
    r["skew"] = torch.randn(e, device="cuda", generator=gen) if case.get("skew") else None
    r["shared_gate"] = (torch.randn((1, d), device="cuda", generator=gen) * STD).to(torch.bfloat16)
    return r


def _hidden(case: dict, seed: int) -> torch.Tensor:
    """Normalised hidden states, [layers, n, hidden] bf16."""
    d = SHAPES[case["shape"]]["hidden"]
    return torch.randn((case.get("layers", 1), case["n"], d), device="cuda",
                       generator=_gen(seed, 1)).to(torch.bfloat16)


def _seam_ids(case: dict, seed: int) -> torch.Tensor:
    """Distinct expert ids per token, unevenly popular."""
    sh = SHAPES[case["shape"]]
    gen = _gen(seed, 5)
    pop = torch.randn(sh["experts"], device="cuda", generator=gen) * 0.5
    z = pop - torch.log(-torch.log(torch.rand((case["n"], sh["experts"]), device="cuda",
                                              generator=gen).clamp_(1e-9, 1 - 1e-7)))
    return torch.topk(z, sh["k"], dim=-1).indices.to(torch.int32)


def _glu(case: dict, seed: int, layer: int):
    from pagedmoe_amd.streaming import QuantizedSwitchGLU
    sh = SHAPES[case["shape"]]
    glu = QuantizedSwitchGLU(sh["hidden"], sh["inter"], sh["experts"], sh["bits"],
                             n_shared=sh["shared"])
    _fill(glu.slab, sh, seed, layer)
    return glu


def _moe(case: dict, seed: int, layer: int):
    from pagedmoe_amd.streaming import SigmoidGroupMoEBlock, SoftmaxMoEBlock
    sh = SHAPES[case["shape"]]
    r = _router(case, seed, layer)
    glu = _glu(case, seed, layer)
    if sh["scoring"] == "sigmoid":
        return SigmoidGroupMoEBlock(r["gate"], r["bias"], glu, sh["k"], N_GROUP, TOPK_GROUP,
                                    ROUTED_SCALE)
    return SoftmaxMoEBlock(r["gate"], glu, sh["k"], logit_bias=r["skew"],
                           shared_expert_gate=r["shared_gate"] if sh["shared"] else None)


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    if kind == "format":
        w = torch.randn((case["rows"], case["cols"]), device="cuda", generator=_gen(seed, 9)) * STD
        return {"case": case, "w": w}
    x = _hidden(case, seed)
    if kind == "seam":
        return {"case": case, "x": x[0], "inds": _seam_ids(case, seed), "glu": _glu(case, seed, 0)}
    blocks = torch.nn.ModuleList(_moe(case, seed, li) for li in range(case["layers"]))
    state = {"case": case, "x": x, "blocks": blocks}
    if kind == "paged":
        from pagedmoe_amd.streaming import build_cache_for, patch_model
        e = SHAPES[case["shape"]]["experts"]
        slots = case["slots"] or (e * case["layers"] * 5) // 8
        cache = build_cache_for(blocks, slots)
        # prediction off: its governor alternates it on and off while it learns
        patch_model(blocks, cache, predict_mode="off")
    return state


# ---------------------------------------------------------------- one pass

def run(state: dict):
    case = state["case"]
    kind = case["kind"]
    if kind == "format":
        from pagedmoe_amd import kernels
        q, s, b = kernels.quantize(state["w"], case["bits"])
        return {"q": q, "scales": s, "biases": b,
                "w": kernels.dequant(q, s, b, case["bits"])}
    if kind == "seam":
        return {"y": state["glu"](state["x"], state["inds"])}
    out = []
    if kind == "paged":
        for t in range(case["n"]):
            for li, blk in enumerate(state["blocks"]):
                out.append(_call(blk, state["x"][li, t:t + 1]))
        return out
    for li, blk in enumerate(state["blocks"]):
        out.append(_call(blk, state["x"][li]))
    return out


def _call(blk, x):
    y = blk(x)
    inds, weights = blk.last_routing
    return {"out": y, "inds": inds, "weights": weights}


# ---------------------------------------------------------------- what it cannot do without

def work(case: dict) -> dict:
    if case["kind"] == "format":
        vals = case["rows"] * case["cols"]
        packed = vals * case["bits"] // 8 + vals // 64 * 4
        return {"bytes": 4 * vals + 2 * packed + 2 * vals, "flops": 8 * vals}
    sh = SHAPES[case["shape"]]
    d, i, e, k = sh["hidden"], sh["inter"], sh["experts"], sh["k"]
    per = 3 * d * i * sh["bits"] // 8 + 3 * d * i // 64 * 4
    n, layers = case["n"], case.get("layers", 1)
    # a paged pass is n tokens, one after the other
    tokens, calls = (1, n) if case["kind"] == "paged" else (n, 1)
    seen = e * (1.0 - (1.0 - k / e) ** tokens) + (sh["shared"] if case["kind"] != "seam" else 0)
    rows = tokens * (k + (sh["shared"] if case["kind"] != "seam" else 0))
    if case["kind"] == "seam":
        io = 2 * tokens * d * (1 + k) + 4 * tokens * k
        flops = 6.0 * d * i * rows
    else:
        io = 4 * tokens * d + 8 * tokens * k + 2 * e * d
        flops = 6.0 * d * i * rows + 2.0 * tokens * d * e
    return {"bytes": int(layers * calls * (seen * per + io)), "flops": int(layers * calls * flops)}


def tolerance(case: dict):
    if case["kind"] == "format":
        return "exact"  # codes, bf16 scales and biases, and the bf16 values they stand for
    # bf16 outputs over a bf16 SwiGLU intermediate and fp32 sums
    return {"rel": 1e-2}


# ---------------------------------------------------------------- 64 bits

def exact(case: dict, seed: int):
    if case["kind"] == "format":
        return _exact_format(case, seed)
    sh = SHAPES[case["shape"]]
    x = _hidden(case, seed)
    outs = []
    for li in range(case.get("layers", 1)):
        xl = x[li].double()
        if case["kind"] == "seam":
            inds, wts = _seam_ids(case, seed).long(), None
        else:
            inds, wts = _exact_route(case, seed, li, xl)
        y = _exact_experts(case, seed, li, xl, inds, wts)
        outs.append({"y": y} if wts is None else {"out": y, "inds": None, "weights": wts})
    if case["kind"] == "seam":
        return outs[0]
    if case["kind"] == "paged":
        return [{"out": o["out"][t:t + 1], "inds": None, "weights": o["weights"][t:t + 1]}
                for t in range(case["n"]) for o in outs]
    return outs


def _exact_route(case: dict, seed: int, layer: int, x: torch.Tensor):
    sh = SHAPES[case["shape"]]
    r = _router(case, seed, layer)
    logits = x @ r["gate"].double().T
    if sh["scoring"] == "softmax":
        if r["skew"] is not None:
            logits = logits + r["skew"].double()
        p, inds = torch.topk(torch.softmax(logits, -1), sh["k"], dim=-1)
        return inds, p / p.sum(-1, keepdim=True)
    sig = torch.sigmoid(logits)
    c = (sig + r["bias"].double()).reshape(x.shape[0], N_GROUP, -1)
    keep = torch.topk(torch.topk(c, 2, dim=-1).values.sum(-1), TOPK_GROUP, dim=-1).indices
    mask = torch.zeros(c.shape[:2], dtype=torch.bool, device=x.device).scatter_(1, keep, True)
    c = torch.where(mask[..., None], c, torch.zeros_like(c)).reshape(x.shape[0], -1)
    inds = torch.topk(c, sh["k"], dim=-1).indices
    p = sig.gather(1, inds)
    return inds, p / p.sum(-1, keepdim=True) * ROUTED_SCALE


def _exact_experts(case: dict, seed: int, layer: int, x, inds, wts):
    """Combined outputs [n, hidden], or per-slot ones [n, k, hidden] when no
    weights are given."""
    sh = SHAPES[case["shape"]]
    n, d = x.shape
    out = torch.zeros((n, d) if wts is not None else (n, sh["k"], d), dtype=torch.float64,
                      device=x.device)

    def ffn(part, j, rows):
        def weight(proj):
            q, s, b = (t[j] for t in part[proj])
            g = q.double().reshape(q.shape[0], -1, 64)
            return (g * s.double()[..., None] + b.double()[..., None]).reshape(q.shape)
        h = rows @ weight("gate_proj").T
        h = h * torch.sigmoid(h) * (rows @ weight("up_proj").T)
        return h @ weight("down_proj").T

    used = set(torch.unique(inds).tolist())
    for e0, part in _expert_chunks(sh, seed, layer):
        for j in range(part["gate_proj"][0].shape[0]):
            e = e0 + j
            if e in used:
                tok, col = (inds == e).nonzero(as_tuple=True)
                y = ffn(part, j, x[tok])
                if wts is None:
                    out[tok, col] = y
                else:
                    out.index_add_(0, tok, y * wts[tok, col][:, None])
            elif e == sh["experts"] and wts is not None:
                y = ffn(part, j, x)
                if sh["scoring"] == "softmax":
                    gate = _router(case, seed, layer)["shared_gate"].double()
                    y = y * torch.sigmoid(x @ gate.T)
                out += y
    return out


def _exact_format(case: dict, seed: int):
    w = torch.randn((case["rows"], case["cols"]), device="cuda", generator=_gen(seed, 9)) * STD
    top = (1 << case["bits"]) - 1
    g = w.reshape(case["rows"], -1, 64)
    lo, hi = g.amin(-1), g.amax(-1)
    s = ((hi - lo) / top).to(torch.bfloat16).double()
    s = torch.where(s == 0, torch.ones_like(s), s)[..., None]
    b = lo.to(torch.bfloat16).double()[..., None]
    q = torch.round((g.double() - b) / s).clamp_(0, top)
    return {"q": None, "scales": None, "biases": None, "w": (q * s + b).reshape(w.shape)}
