"""Timed cases: the work a user of weightstream_amd has it do, through launch.py.

A case is a dict of plain values; `kind` names the work:

  decode   ws_moe_decode_route for `tokens` successive tokens (routing, the
           eight or six routed FP4 experts, the ordered sum), captured in a HIP
           graph as a serving loop captures its decode step. Every token has
           experts of its own, so their weights come from HBM.
  layer    one whole MoE block for a batch of `m` sequences: FP8 out-projection
           with the residual add, f32 gate, top-k, routed FP4 experts, shared
           FP8 expert, captured in a HIP graph.
  prefill  top-k and the routed experts for `m` tokens of a prompt.
  gate     gate logits and top-k for `m` tokens.
  linear   one FP8 (or FP4) linear: the activation's quantisation and the GEMM.
  shared   the shared FP8 expert for `m` tokens (w1 and w3 in one matrix).
  encode   checkpoint ingest: f32 weights to FP4 in the packed expert layout,
           or to FP8 with 32x32 scales.

Weights are N(0, 0.02) and activations N(0, 1), 1% of a linear's activations 20
times larger; both come from the seed alone.
"""
import math

import torch

from weightstream_amd import launch as L

DEV = "cuda:0"
LIMIT = 10.0   # swiglu_limit

# the two MoE layers this repository is configured for: the benchmark's
# (384 experts, top-8, sigmoid) and DS4.1F's (top-6, sqrtsoftplus)
BLOCK = {"dim": 4096, "inter": 2048, "experts": 384, "top_k": 8, "score": "sigmoid", "scale": 1.0}
DS = {"dim": 5120, "inter": 2304, "experts": 384, "top_k": 6, "score": "sqrtsoftplus",
      "scale": 1.5}
# (N, K) of the engine's FP8 projections, with their ws_fp8_gemm_tl kinds
PROJECTIONS = [(1280, 5120, L.TL_QA), (8192, 1280, L.TL_QB), (512, 5120, L.TL_WKV),
               (2048, 4096, L.TL_WO_A), (5120, 2048, L.TL_WO_B), (2304, 5120, L.TL_SHARED_W13),
               (4608, 5120, L.TL_SHARED_W13_FUSED), (5120, 2304, L.TL_SHARED_W2),
               (25600, 5120, L.TL_ENGRAM_WKV), (1280, 15360, L.TL_DRAFTER_MAIN_PROJ)]
FORMATS = ("fp8", "fp8_bf16", "f32s", "f32s_bf16", "fp4", "tl")


def listed():
    return [
        # single-stream generation: the routed experts of 8 successive tokens
        dict(BLOCK, name="decode_8_tokens", kind="decode", tokens=8),
        # the whole block at the batch sizes of generation: one sequence, and
        # the odd number that a continuous batch holds at a given moment
        dict(BLOCK, name="layer_m1", kind="layer", m=1, out_k=8192, shared=2048),
        dict(BLOCK, name="layer_m27", kind="layer", m=27, out_k=8192, shared=2048),
        # a short prompt with skewed expert popularity
        dict(BLOCK, name="prefill_132_zipf", kind="prefill", m=132, zipf=1.1),
        # a ragged prompt of the other layer, popularity nearly even
        dict(DS, name="prefill_600_ds", kind="prefill", m=600, zipf=0.3),
        # a long prompt (or several packed together): the largest call
        dict(BLOCK, name="prefill_4096", kind="prefill", m=4096, zipf=0.5),
        # routing of a prompt
        dict(BLOCK, name="gate_1024", kind="gate", m=1024, gate="f32"),
        # one token through one small projection: launches and latency
        dict(name="linear_m1_q_a", kind="linear", m=1, n=1280, k=5120, fmt="fp8"),
        # the 128-token GEMM with the f32 block scales of such checkpoints
        dict(name="linear_m128_f32s", kind="linear", m=128, n=4096, k=4096, fmt="f32s_bf16"),
        # a long prompt through the attention output projection
        dict(name="linear_m4096_out", kind="linear", m=4096, n=4096, k=8192, fmt="fp8_bf16"),
        # the shared expert over a ragged prompt
        dict(name="shared_m777_ds", kind="shared", m=777, dim=5120, inter=2304),
        # ingest of the gate matrices of 16 experts
        dict(name="encode_fp4_experts", kind="encode", rows=16 * 2304, cols=5120, fmt="fp4"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _layer_shape(rng):
    """One of the two layers, or a smaller one with sizes of its own."""
    kind = rng.randrange(4)
    if kind < 3:
        return dict(BLOCK if kind < 2 else DS)
    return {"dim": 256 * rng.randint(4, 20), "inter": 128 * rng.randint(4, 20),
            "experts": rng.choice([48, 64, 96, 128, 160, 256]), "top_k": rng.choice([4, 6, 8]),
            "score": rng.choice(["sigmoid", "sqrtsoftplus"]), "scale": rng.choice([1.0, 1.5])}


def draw(rng):
    kind = rng.choice(["decode", "layer", "layer", "prefill", "prefill", "prefill", "gate",
                       "linear", "linear", "linear", "shared", "encode"])
    if kind == "decode":
        return dict(_layer_shape(rng), kind=kind, tokens=rng.randint(4, 12))
    if kind == "layer":
        return dict(_layer_shape(rng), kind=kind, m=_log(rng, 1, 64),
                    out_k=rng.choice([4096, 8192]), shared=256 * rng.randint(4, 9))
    if kind == "prefill":
        return dict(_layer_shape(rng), kind=kind, m=_log(rng, 65, 4000),
                    zipf=round(rng.uniform(0.0, 1.2), 2))
    if kind == "gate":
        return dict(_layer_shape(rng), kind=kind, m=_log(rng, 1, 4096),
                    gate=rng.choice(["f32", "bf16"]))
    if kind == "shared":
        return {"kind": kind, "m": _log(rng, 1, 4096), "dim": 256 * rng.randint(8, 20),
                "inter": 128 * rng.randint(8, 18)}
    if kind == "encode":
        return {"kind": kind, "rows": 32 * _log(rng, 16, 1500), "cols": 128 * rng.randint(8, 40),
                "fmt": rng.choice(["fp4", "fp8"])}
    fmt = rng.choice(FORMATS)
    n, k, _ = rng.choice(PROJECTIONS)
    if fmt != "tl" and rng.random() < 0.5:
        n, k = 16 * _log(rng, 16, 1024), 128 * _log(rng, 8, 80)
    return {"kind": kind, "m": _log(rng, 1, 4096), "n": n, "k": k, "fmt": fmt}


# ---- inputs, in plain torch -------------------------------------------------
def _gen(seed):
    gen = torch.Generator(device=DEV)
    gen.manual_seed(int(seed))
    return gen


def _normal(gen, *shape, std=1.0):
    return torch.empty(shape, dtype=torch.float32, device=DEV).normal_(0.0, std, generator=gen)


def _ceil_log2(x):
    m, e = torch.frexp(x)
    return torch.where(m > 0.5, e, e - 1)


def _over(x, n):
    """x / n, correctly rounded (a division by a Python number multiplies by
    its reciprocal)."""
    return x / torch.full((), n, dtype=x.dtype, device=x.device)


def _fp4_weights(gen, rows, cols):
    """N(0, 0.02) as packed e2m1 (low nibble = even column) and UE8M0 scales
    per 1x32."""
    q = torch.empty((rows, cols // 2), dtype=torch.uint8, device=DEV)
    s = torch.empty((rows, cols // 32), dtype=torch.uint8, device=DEV)
    mids = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device=DEV)
    step = max(1, (1 << 27) // cols)
    for r in range(0, rows, step):
        w = _normal(gen, min(step, rows - r), cols // 32, 32, std=0.02)
        e = _ceil_log2(_over(w.abs().amax(-1), 6.0))
        s[r:r + step] = (e + 127).to(torch.uint8)
        w = torch.ldexp(w, -e[..., None])
        code = torch.bucketize(w.abs(), mids, out_int32=True).to(torch.uint8)
        code |= (w < 0).to(torch.uint8) << 3
        code = code.view(code.shape[0], cols)
        q[r:r + step] = code[:, 0::2] | (code[:, 1::2] << 4)
    return q, s


def _fp8_weights(gen, rows, cols, f32_scales=False):
    """N(0, 0.02) as e4m3 with UE8M0 scales per 32x32, or f32 ones per 128x128."""
    b = 128 if f32_scales else 32
    pad = -rows % b
    w = torch.nn.functional.pad(_normal(gen, rows, cols, std=0.02), (0, 0, 0, pad))
    w = w.view((rows + pad) // b, b, cols // b, b)
    amax = w.abs().amax((1, 3)).clamp_min(1e-4)
    if f32_scales:
        s = _over(amax, 448.0)
        w = w / s[:, None, :, None]
    else:
        e = _ceil_log2(_over(amax, 448.0))
        s = (e + 127).to(torch.uint8)
        w = torch.ldexp(w, -e[:, None, :, None])
    q = w.clamp(-448, 448).view(rows + pad, cols)[:rows].to(torch.float8_e4m3fn)
    return q.view(torch.uint8).contiguous(), s


def _moe_weights(gen, c):
    E, dim, inter = c["experts"], c["dim"], c["inter"]
    return (_fp4_weights(gen, E * inter, dim) + _fp4_weights(gen, E * inter, dim)
            + _fp4_weights(gen, E * dim, inter))


def _inputs(c, seed):
    gen = _gen(seed)
    kind = c["kind"]
    if kind in ("decode", "prefill"):
        m, E = c["tokens"] if kind == "decode" else c["m"], c["experts"]
        logits = _normal(gen, m, E)
        if kind == "prefill":
            rank = torch.randperm(E, device=DEV, generator=gen) + 1
            logits = logits - c["zipf"] * torch.log(rank.float())
        return {"logits": logits, "bias": _normal(gen, E, std=0.1), "x": _normal(gen, m, c["dim"]),
                "routed": _moe_weights(gen, c)}
    if kind == "layer":
        return {"attn": _normal(gen, c["m"], c["out_k"]), "h0": _normal(gen, c["m"], c["dim"]),
                "wo": _fp8_weights(gen, c["dim"], c["out_k"]),
                "gate": _normal(gen, c["experts"], c["dim"], std=0.02),
                "bias": _normal(gen, c["experts"], std=0.1), "routed": _moe_weights(gen, c),
                "w13": _fp8_weights(gen, 2 * c["shared"], c["dim"]),
                "w2": _fp8_weights(gen, c["dim"], c["shared"])}
    if kind == "gate":
        gate = _normal(gen, c["experts"], c["dim"], std=0.02)
        return {"x": _normal(gen, c["m"], c["dim"]), "bias": _normal(gen, c["experts"], std=0.1),
                "gate": gate if c["gate"] == "f32" else gate.bfloat16()}
    if kind == "linear":
        x = _normal(gen, c["m"], c["k"])
        x = torch.where(torch.rand(x.shape, device=DEV, generator=gen) < 0.01, x * 20, x)
        if c["fmt"] == "fp4":
            return {"x": x, "w": _fp4_weights(gen, c["n"], c["k"])}
        return {"x": x, "w": _fp8_weights(gen, c["n"], c["k"], c["fmt"].startswith("f32s"))}
    if kind == "shared":
        return {"x": _normal(gen, c["m"], c["dim"]),
                "w13": _fp8_weights(gen, 2 * c["inter"], c["dim"]),
                "w2": _fp8_weights(gen, c["dim"], c["inter"])}
    return {"w": _normal(gen, c["rows"], c["cols"], std=0.02)}


# ---- the framework's side ------------------------------------------------------
_splitk = {}       # split-K workspace per stream, as a program registers it once
_capture = None    # the stream that graphs are captured on


def _split_k_workspace(stream, shapes):
    need = max([256] + [L.gemm_workspace_size(*s) for s in shapes])
    have = _splitk.get(stream.cuda_stream)
    if have is None or have.numel() < need:
        have = torch.empty(need, dtype=torch.uint8, device=DEV)
        L.set_gemm_workspace(have, stream=stream)
        _splitk[stream.cuda_stream] = have
    return have


def _bytes(n):
    return torch.empty(int(n), dtype=torch.uint8, device=DEV)


def _f32(*shape):
    return torch.empty(shape, dtype=torch.float32, device=DEV)


def _pack(c, raw):
    E, dim, inter = c["experts"], c["dim"], c["inter"]
    return (L.prepack_fp4_new(raw[0], raw[1], E * inter, dim)
            + L.prepack_fp4_new(raw[2], raw[3], E * inter, dim)
            + L.prepack_fp4_new(raw[4], raw[5], E * dim, inter))


SCORES = {"sigmoid": L.SCORE_SIGMOID, "sqrtsoftplus": L.SCORE_SQRTSOFTPLUS}


def prepare(case, seed):
    c, s = case, _inputs(case, seed)
    s["case"], kind = c, c["kind"]
    if "experts" in c:
        rows = c["tokens"] if kind == "decode" else c["m"]
        s["idx"] = torch.empty((rows, c["top_k"]), dtype=torch.int32, device=DEV)
        s["wts"] = _f32(rows, c["top_k"])
    if kind in ("decode", "prefill", "layer"):
        s["routed"] = _pack(c, s["routed"])
        s["y"] = _f32(rows, c["dim"])
        s["dws"] = _bytes(L.moe_decode_workspace_size(c["dim"], c["inter"], c["top_k"]))
    if kind == "prefill" or kind == "layer" and c["m"] > 1:
        s["pws"] = _bytes(L.moe_prefill_workspace_size(c["m"], c["dim"], c["inter"], c["top_k"],
                                                       c["experts"]))
    if kind in ("layer", "shared"):
        inter = c["shared"] if kind == "layer" else c["inter"]
        s["sws"] = _bytes(L.shared_expert_workspace_size(c["m"], c["dim"], inter))
        shapes = [(c["m"], 2 * inter, c["dim"]), (c["m"], c["dim"], inter)]
    if kind == "layer":
        shapes.append((c["m"], c["dim"], c["out_k"]))
        s["h"] = _f32(c["m"], c["dim"])
        s["aq"], s["as"] = _bytes(c["m"] * c["out_k"]), _bytes(c["m"] * c["out_k"] // 32)
        s["hs"], s["ys"] = _f32(c["m"], c["shared"]), _f32(c["dim"])
    if kind in ("gate", "layer"):
        s["logits"] = _f32(c["m"], c["experts"])
    if kind == "shared":
        s["y"] = _f32(c["m"], c["dim"])
        s["splitk"] = _split_k_workspace(torch.cuda.current_stream(), shapes)
    if kind == "linear":
        m, n, k, fmt = c["m"], c["n"], c["k"], c["fmt"]
        s["q"] = _bytes(m * k)
        if fmt.startswith("f32s"):
            s["s"] = _f32(m, k // 128)
        elif fmt == "tl":
            # the scale bytes, and their packed words from the next multiple of 16
            words = (m * k // 32 + 15) // 16 * 16
            both = _bytes(words + m * k // 32)
            s["s"], s["words"] = both, both[words:]
            s["kind"] = {(pn, pk): kind for pn, pk, kind in PROJECTIONS}[(n, k)]
            s["w"] = (s["w"][0], s["w"][1].repeat_interleave(32, 0)[:n].contiguous())
        else:
            s["s"] = _bytes(m * k // 32)
        s["y"] = torch.empty((m, n), device=DEV,
                             dtype=torch.bfloat16 if fmt.endswith("bf16") else torch.float32)
        s["splitk"] = _split_k_workspace(torch.cuda.current_stream(), [(m, n, k)])
    if kind == "encode":
        rows, cols = c["rows"], c["cols"]
        if c["fmt"] == "fp4":
            s["q"], s["s"] = _bytes(rows * cols // 2), _bytes(rows * cols // 32)
            s["pq"], s["ps"] = _bytes(rows * cols // 2), _bytes(L.packed_fp4_scale_bytes(rows, cols))
        else:
            s["q"], s["s"] = _bytes(rows * cols), _bytes((rows + 31) // 32 * (cols // 32))
    if kind in ("decode", "layer"):
        _capture_step(s, _decode if kind == "decode" else _layer,
                      shapes if kind == "layer" else [])
    return s


def _capture_step(s, step, shapes):
    global _capture
    if _capture is None:
        _capture = torch.cuda.Stream()
    s["splitk"] = _split_k_workspace(_capture, shapes)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(_capture):
        step(s)
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=_capture):
            step(s)
    torch.cuda.synchronize()
    s["graph"] = graph


def _decode(s):
    c = s["case"]
    for t in range(c["tokens"]):
        L.moe_decode_route(s["logits"][t], s["bias"], SCORES[c["score"]], 1.0, 1, c["scale"],
                           s["x"][t], *s["routed"], s["y"][t], s["idx"][t], s["wts"][t], c["dim"],
                           c["inter"], c["experts"], c["top_k"], s["dws"], swiglu_limit=LIMIT)


def _layer(s):
    c = s["case"]
    m, dim, inter, E, k, si = (c["m"], c["dim"], c["inter"], c["experts"], c["top_k"], c["shared"])
    h, score = s["h"], SCORES[c["score"]]
    h.copy_(s["h0"])
    if m == 1:
        L.fp8_gemv_acc(s["attn"], *s["wo"], h, m, dim, c["out_k"])
        L.moe_gate_shared_w13(h, s["gate"], s["logits"], *s["w13"], s["hs"], m, dim, E, si,
                              swiglu_limit=LIMIT)
        L.moe_decode_route_shared(s["logits"], s["bias"], score, 1.0, 1, c["scale"], h,
                                  *s["routed"], s["y"], s["idx"], s["wts"], dim, inter, E, k,
                                  s["hs"], *s["w2"], si, s["ys"], h, s["dws"], swiglu_limit=LIMIT)
        return
    L.emit8(s["attn"], s["aq"], s["as"], m * c["out_k"])
    L.fp8_gemm_acc(s["aq"], s["as"], *s["wo"], h, m, dim, c["out_k"])
    L.moe_gate_logits(h, s["gate"], s["logits"], m, dim, E)
    L.moe_topk(s["logits"], s["bias"], None, s["idx"], s["wts"], m, E, k, score, 1.0, True,
               c["scale"])
    L.moe_prefill(h, s["idx"], s["wts"], *s["routed"], s["y"], m, dim, inter, E, k, s["pws"],
                  swiglu_limit=LIMIT)
    L.shared_expert_fp8_w13_acc(h, *s["w13"], *s["w2"], s["y"], h, m, dim, si, s["sws"],
                                swiglu_limit=LIMIT)


def _linear(s):
    c = s["case"]
    m, n, k, fmt = c["m"], c["n"], c["k"], c["fmt"]
    x, q, sc, (w, ws), y = s["x"], s["q"], s["s"], s["w"], s["y"]
    if fmt.startswith("f32s"):
        L.act_quant_f32s(x, q, sc, m, k)
        L.fp8_gemm_f32s(q, sc, w, ws, y, m, n, k, out_bf16=fmt == "f32s_bf16")
    elif fmt == "tl":
        L.emit8_packed(x, q, sc, m * k)
        L.fp8_gemm_tl(s["kind"], q, s["words"], w, ws, y, m)
    else:
        L.emit8(x, q, sc, m * k)
        gemm = {"fp8": L.fp8_gemm, "fp8_bf16": L.fp8_gemm_bf16, "fp4": L.fp4_gemm}[fmt]
        gemm(q, sc, w, ws, y, m, n, k)
    return y


def run(state):
    s, c = state, state["case"]
    kind = c["kind"]
    if kind in ("decode", "layer"):
        s["graph"].replay()
        return {"y": s["y" if kind == "decode" else "h"], "idx": s["idx"], "weights": s["wts"]}
    if kind == "linear":
        return _linear(s)
    if kind == "shared":
        L.shared_expert_fp8_w13(s["x"], *s["w13"], *s["w2"], s["y"], c["m"], c["dim"], c["inter"],
                                s["sws"], swiglu_limit=LIMIT)
        return s["y"]
    if kind == "encode":
        L_quant = L.weight_quant_fp4 if c["fmt"] == "fp4" else L.weight_quant_fp8
        L_quant(s["w"], s["q"], s["s"], c["rows"], c["cols"])
        if c["fmt"] == "fp8":
            return s["q"], s["s"]
        L.prepack_fp4(s["q"], s["s"], c["rows"], c["cols"], s["pq"], s["ps"])
        return s["pq"], s["ps"]
    if kind == "gate":
        L.moe_gate_logits(s["x"], s["gate"], s["logits"], c["m"], c["dim"], c["experts"])
    L.moe_topk(s["logits"], s["bias"], None, s["idx"], s["wts"], c["m"], c["experts"], c["top_k"],
               SCORES[c["score"]], 1.0, True, c["scale"])
    out = {"idx": s["idx"], "weights": s["wts"]}
    if kind == "gate":
        return dict(out, logits=s["logits"])
    L.moe_prefill(s["x"], s["idx"], s["wts"], *s["routed"], s["y"], c["m"], c["dim"], c["inter"],
                  c["experts"], c["top_k"], s["pws"], swiglu_limit=LIMIT)
    return dict(out, y=s["y"])


# ---- what a pass cannot do without ------------------------------------------------
def _touched(c, m, std=1.0):
    """Experts that m tokens reach, in one draw of the case's distributions."""
    gen = torch.Generator()
    gen.manual_seed(1)
    E = c["experts"]
    rank = torch.arange(1, E + 1, dtype=torch.float32)
    v = torch.empty(m, E).normal_(generator=gen) * std - c.get("zipf", 0.0) * torch.log(rank)
    s = torch.sigmoid(v) if c["score"] == "sigmoid" else torch.nn.functional.softplus(v).sqrt()
    s = s + 0.1 * torch.empty(E).normal_(generator=gen)
    return len(torch.unique(torch.topk(s, c["top_k"], dim=-1).indices))


def _moe_work(c, m, experts):
    mat = c["dim"] * c["inter"] * 17 // 32
    return experts * 3 * mat, 6.0 * m * c["top_k"] * c["dim"] * c["inter"]


def work(case):
    c, kind = case, case["kind"]
    if kind == "decode":
        b, f = _moe_work(c, c["tokens"], c["tokens"] * c["top_k"])
        return {"bytes": b + c["tokens"] * (8 * c["dim"] + 4 * c["experts"]), "flops": f}
    if kind == "prefill":
        b, f = _moe_work(c, c["m"], _touched(c, c["m"]))
        return {"bytes": b + c["m"] * (8 * c["dim"] + 4 * c["experts"]), "flops": f}
    if kind == "gate":
        size = 4 if c["gate"] == "f32" else 2
        return {"bytes": 4 * c["m"] * (c["dim"] + c["experts"]) + size * c["dim"] * c["experts"],
                "flops": 2.0 * c["m"] * c["dim"] * c["experts"]}
    if kind == "layer":
        m, dim = c["m"], c["dim"]
        std = 0.02 * math.sqrt(dim * (1 + 0.02 ** 2 * c["out_k"]))   # of the gate logits
        b, f = _moe_work(c, m, _touched(c, m, std))
        fp8 = dim * c["out_k"] + 3 * dim * c["shared"]
        return {"bytes": b + fp8 * 1025 // 1024 + 4 * dim * c["experts"]
                + 4 * m * (c["out_k"] + 2 * dim),
                "flops": f + 2.0 * m * (fp8 + dim * c["experts"])}
    if kind == "linear":
        m, n, k = c["m"], c["n"], c["k"]
        out = 2 if c["fmt"].endswith("bf16") else 4
        return {"bytes": 4 * m * k + (n * k * 17 // 32 if c["fmt"] == "fp4" else n * k) + out * m * n,
                "flops": 2.0 * m * n * k}
    if kind == "shared":
        m, dim, inter = c["m"], c["dim"], c["inter"]
        return {"bytes": 8 * m * dim + 3 * dim * inter, "flops": 6.0 * m * dim * inter}
    n = c["rows"] * c["cols"]
    return {"bytes": 4 * n + (n * 17 // 32 if c["fmt"] == "fp4" else n), "flops": 0}


def tolerance(case):
    kind = case["kind"]
    if kind in ("gate", "encode"):
        return "exact"   # sequential f32 sums and bytes, by contract
    if kind == "linear":
        # f32 sums of up to 15360 products in another order; bf16 results
        # differ where such a sum crosses a rounding boundary
        return {"rel": 1e-3, "max": 1e-2} if case["fmt"].endswith("bf16") else {"rel": 2e-6, "max": 2e-5}
    # an h within f32 rounding of an e4m3 midpoint may land one step apart
    return {"rel": 1e-3, "max": 3e-2, "differ": 1e-3}


# ---- the same results in 64 bits, in plain torch ------------------------------------
_E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, 0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0)


def _pow2(s):
    return torch.ldexp(torch.ones((), dtype=torch.float64, device=DEV), s.int() - 127)


def _fp4_values(q, s):
    lut = torch.tensor(_E2M1, dtype=torch.float64, device=DEV)
    v = torch.stack((lut[(q & 15).int()], lut[(q >> 4).int()]), -1).view(q.shape[0], -1, 32)
    return (v * _pow2(s)[..., None]).view(q.shape[0], -1)


def _fp8_values(q, s):
    v = q.view(torch.float8_e4m3fn).double()
    b = 32 if s.dtype == torch.uint8 else 128
    s = _pow2(s) if s.dtype == torch.uint8 else s.double()
    return v * s.repeat_interleave(b, 0)[:v.shape[0]].repeat_interleave(b, 1)


def _e4m3(v):
    """Values on the e4m3 grid; the format's encoder writes the code of 1 for
    what rounds up to 2^-6 from below."""
    r = v.float().clamp(-448, 448).to(torch.float8_e4m3fn).double()
    return torch.where((v.abs() < 2.0 ** -6) & (r.abs() == 2.0 ** -6), torch.sign(v).double(), r)


def _quantised(x, f32_scales=False):
    """x after the 1x32 UE8M0 (or 1x128 f32) FP8 quantisation."""
    b = x.view(x.shape[0], -1, 128 if f32_scales else 32)
    amax = b.abs().amax(-1, keepdim=True).clamp_min(1e-4)
    if f32_scales:
        s = _over(amax, 448.0)
        return (_e4m3(b / s) * s.double()).view(x.shape)
    s = torch.ldexp(torch.ones_like(amax), _ceil_log2(_over(amax, 448.0)))
    return (_e4m3(b / s) * s.double()).view(x.shape)


def _swiglu(g, u, w=1.0):
    return torch.nn.functional.silu(g.clamp(max=LIMIT)) * u.clamp(-LIMIT, LIMIT) * w


def _route(c, logits, bias):
    v = logits.double()
    s = torch.sigmoid(v) if c["score"] == "sigmoid" else torch.nn.functional.softplus(v).sqrt()
    idx = torch.topk(s + bias.double(), c["top_k"], dim=-1).indices
    w = s.gather(1, idx)
    return idx, w / (w.sum(-1, keepdim=True) + 1e-20) * c["scale"]


def _experts(c, raw, x, idx, w):
    dim, inter = c["dim"], c["inter"]
    q = _quantised(x)
    y = torch.zeros((x.shape[0], dim), dtype=torch.float64, device=DEV)
    for e in torch.unique(idx).tolist():
        token, slot = torch.nonzero(idx == e, as_tuple=True)
        gu, dn = slice(e * inter, (e + 1) * inter), slice(e * dim, (e + 1) * dim)
        g = q[token] @ _fp4_values(raw[0][gu], raw[1][gu]).T
        u = q[token] @ _fp4_values(raw[2][gu], raw[3][gu]).T
        h = _quantised(_swiglu(g, u, w[token, slot][:, None]))
        y.index_add_(0, token, h @ _fp4_values(raw[4][dn], raw[5][dn]).T)
    return y


def _shared_expert(x, w13, w2):
    g, u = (_quantised(x) @ _fp8_values(*w13).T).chunk(2, 1)
    return _quantised(_swiglu(g, u)) @ _fp8_values(*w2).T


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "encode":
        return None   # bytes only
    i = _inputs(c, seed)
    if kind == "linear":
        q = _quantised(i["x"], c["fmt"].startswith("f32s"))
        return q @ (_fp4_values(*i["w"]) if c["fmt"] == "fp4" else _fp8_values(*i["w"])).T
    if kind == "shared":
        return _shared_expert(i["x"], i["w13"], i["w2"])
    if kind == "gate":
        logits = i["x"].double() @ i["gate"].double().T
        return {"idx": None, "weights": None, "logits": logits}
    if kind == "layer":
        h = i["h0"].double() + _quantised(i["attn"]) @ _fp8_values(*i["wo"]).T
        idx, w = _route(c, h @ i["gate"].double().T, i["bias"])
        y = _experts(c, i["routed"], h, idx, w) + _shared_expert(h, i["w13"], i["w2"])
        return {"y": h + y, "idx": None, "weights": w}
    idx, w = _route(c, i["logits"], i["bias"])
    return {"y": _experts(c, i["routed"], i["x"], idx, w), "idx": None, "weights": w}
