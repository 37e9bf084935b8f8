"""What is timed: the library's work inside a serving program, called through its C ABI with argument structs that the
program keeps, as INTEGRATION.md shows. Four kinds of pass:

  proj     one weight matrix per layer, `n` tokens (1: decode, 2 to 16: small batches and draft verification)
  attn     the projections of an attention layer: q_a, q_b, kv, block-diagonal o_a, o_b (decode to prefill)
  moe      one token through MoE layers: fused router, address table from the chosen ids, expert layer
  prefill  a prompt through one MoE layer: top-6, routing lists, grouped expert GEMMs

Weights are random GGUF blocks with scales that give weights of about 0.02 to 0.04; every layer has its own matrices, so
the pass reads them from HBM as a model of many layers does.
"""
import ctypes as C
import math

import torch

from macseek_amd import _lib, arch
from macseek_amd._lib import MsqBuffer, MsqExpertSlot, MsqMoeDecodeArgs, MsqMoePrefillArgs
from macseek_amd.quant import QType, block_bytes, block_elems, moe_decode_scratch_bytes, moe_prefill_scratch_bytes, row_bytes

DEV = "cuda:0"
TOPK = 6
EPS = 1e-6
DENSE = ("F32", "F16", "BF16")
NORM_FUSED = ("F32", "F16", "BF16", "Q8_0", "Q5_K", "Q6_K", "IQ4_NL")  # types that msq_matvec_rmsnorm takes


def listed():
    return [
        # decode, the smallest matrices of a layer: the KV projection with its input norm, one launch of 2.5 MB a layer
        {"name": "kv_q5k_1tok", "kind": "proj", "t": "Q5_K", "rows": 512, "cols": 7168, "n": 1, "norm": True, "layers": 24},
        # decode, the largest matrix of a model: the output head over a vocabulary of 129280
        {"name": "head_q6k_1tok", "kind": "proj", "t": "Q6_K", "rows": 129280, "cols": 5120, "n": 1, "norm": True, "layers": 1},
        # decode, all projections of an attention layer
        {"name": "attn_q6k_1tok", "kind": "attn", "t": "Q6_K", "dim": 5120, "rank": 1280, "heads": 32768, "kv": 512, "mid": 1024, "n": 1, "layers": 4},
        # four tokens at once: verification of drafted tokens, or four users
        {"name": "attn_q5k_4tok", "kind": "attn", "t": "Q5_K", "dim": 5120, "rank": 1280, "heads": 32768, "kv": 512, "mid": 1024, "n": 4, "layers": 4},
        # sixteen users decoding together, the most that the small-batch entry point takes
        {"name": "attn_q6k_16tok", "kind": "attn", "t": "Q6_K", "dim": 5120, "rank": 1280, "heads": 32768, "kv": 512, "mid": 1024, "n": 16, "layers": 4},
        # a short prompt, or the ragged last chunk of a long one; kv with an odd number of rows
        {"name": "attn_iq4nl_100tok", "kind": "attn", "t": "IQ4_NL", "dim": 4096, "rank": 1536, "heads": 16384, "kv": 577, "mid": 1024, "n": 100, "layers": 1},
        # a full prefill chunk
        {"name": "attn_q6k_2048tok", "kind": "attn", "t": "Q6_K", "dim": 5120, "rank": 1280, "heads": 32768, "kv": 512, "mid": 1024, "n": 2048, "layers": 1},
        # the one-token MoE layer at the benchmark's shape
        {"name": "moe_iq1s_1tok", "kind": "moe", "gu": "IQ1_S", "dn": "IQ1_S", "sh": "IQ2_XXS", "dim": 7168, "inter": 2048, "experts": 384, "layers": 8},
        # the same at the library's default shape with K-quant shared expert
        {"name": "moe_iq2xxs_1tok", "kind": "moe", "gu": "IQ2_XXS", "dn": "IQ2_XXS", "sh": "Q6_K", "dim": 5120, "inter": 2304, "experts": 384, "layers": 8},
        # a short prompt through a MoE layer: most experts get no token or one
        {"name": "prefill_iq1s_37tok", "kind": "prefill", "gu": "IQ1_S", "dn": "IQ1_S", "sh": "Q6_K", "dim": 5120, "inter": 2304, "experts": 384, "n": 37, "zipf": 0.8, "bf16": False},
        # the benchmark's prefill chunk: bf16 activations, skewed expert popularity, no shared expert
        {"name": "prefill_iq2xxs_2048tok", "kind": "prefill", "gu": "IQ2_XXS", "dn": "IQ2_XXS", "sh": "", "dim": 7168, "inter": 2048, "experts": 384, "n": 2048, "zipf": 1.1, "bf16": True},
        # the largest chunk, with shared expert
        {"name": "prefill_iq1s_4096tok", "kind": "prefill", "gu": "IQ1_S", "dn": "IQ1_S", "sh": "Q6_K", "dim": 5120, "inter": 2304, "experts": 384, "n": 4096, "zipf": 0.8, "bf16": False},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("proj", "attn", "attn", "moe", "prefill", "prefill"))
    if kind == "proj":
        t = rng.choice(("Q5_K", "Q6_K", "Q8_0", "IQ1_S", "IQ2_XXS", "IQ4_NL", "BF16", "F16", "F32"))
        rows, cols = _log(rng, 256, 32768), 256 * _log(rng, 4, 40)
        n = 1 if rng.random() < 0.5 else rng.randint(2, 16)
        layers = max(1, min(24, int(4e8 / (_row_bytes(t, cols) * rows))))
        return {"kind": kind, "t": t, "rows": rows, "cols": cols, "n": n, "norm": rng.random() < 0.5, "layers": layers}
    if kind == "attn":
        n = 1 if rng.random() < 0.25 else _log(rng, 2, 2048)
        return {"kind": kind, "t": rng.choice(("Q5_K", "Q6_K", "Q8_0", "IQ4_NL", "IQ2_XXS", "BF16")), "dim": 256 * rng.randint(8, 28),
                "rank": 256 * rng.randint(2, 8), "heads": 2048 * rng.randint(4, 16), "kv": rng.randint(128, 1100), "mid": 128 * rng.randint(2, 9),
                "n": n, "layers": 4 if n <= 16 else 1}
    types = {"gu": rng.choice(("IQ1_S", "IQ2_XXS")), "dn": rng.choice(("IQ1_S", "IQ2_XXS")), "sh": rng.choice(("Q6_K", "Q8_0", "IQ2_XXS", "IQ1_S"))}
    size = {"dim": 256 * rng.randint(8, 28), "inter": 256 * rng.randint(3, 9), "experts": 64 * rng.randint(1, 6)}
    if kind == "moe":
        return {"kind": kind, **types, **size, "layers": 8}
    if rng.random() < 0.3:
        types["sh"] = ""
    return {"kind": kind, **types, **size, "n": _log(rng, 2, 3000), "zipf": rng.choice((0.5, 0.8, 1.1)), "bf16": rng.random() < 0.5}


# ------------------------------------------------------------------------------------------------------------- sizes
def _row_bytes(t, cols):
    return row_bytes(QType[t], cols)


def _attn_shapes(c):
    """(rows, cols, groups) of q_a, q_b, kv, o_a, o_b; o_a is block-diagonal with eight groups over the heads' outputs."""
    return ((c["rank"], c["dim"], 1), (c["heads"], c["rank"], 1), (c["kv"], c["dim"], 1), (8 * c["mid"], c["heads"] // 8, 8), (c["dim"], 8 * c["mid"], 1))


def work(case):
    c = case
    if c["kind"] in ("proj", "attn"):
        n, L = c["n"], c["layers"]
        shapes = _attn_shapes(c) if c["kind"] == "attn" else ((c["rows"], c["cols"], 1),)
        w = sum(_row_bytes(c["t"], cols) * rows for rows, cols, _ in shapes)
        out = sum(rows for rows, _, _ in shapes)
        inp = c["dim"] + c["heads"] + 8 * c["mid"] if c["kind"] == "attn" else c["cols"]
        return {"bytes": L * (w + 4 * n * (inp + out)), "flops": L * 2 * n * sum(rows * cols for rows, cols, _ in shapes)}
    d, i = c["dim"], c["inter"]
    expert = 2 * _row_bytes(c["gu"], d) * i + _row_bytes(c["dn"], i) * d
    shared = 2 * _row_bytes(c["sh"], d) * i + _row_bytes(c["sh"], i) * d if c["sh"] else 0
    if c["kind"] == "moe":
        router = c["experts"] * d * 2
        return {"bytes": c["layers"] * (TOPK * expert + shared + router + 3 * 4 * d), "flops": c["layers"] * 2 * d * (3 * i * (TOPK + 1) + c["experts"])}
    n = c["n"]
    used = _expected_used(c["experts"], n, c["zipf"])
    entries = n * (TOPK + (1 if c["sh"] else 0))
    return {"bytes": used * expert + shared + n * d * (10 if c["bf16"] else 12) + 4 * n * c["experts"], "flops": 2 * 3 * d * i * entries}


def _expected_used(experts, n, zipf):
    """About how many experts get a token (draws with replacement, which is near enough for a byte count)."""
    p = [1.0 / (k + 1) ** zipf for k in range(experts)]
    s = sum(p)
    return int(round(sum(1.0 - (1.0 - v / s) ** (n * TOPK) for v in p)))


def tolerance(case):
    """Largest error against the same path in 64 bits, times about four (measured for every kind and several types).
    One token of a block format has its activations rounded at 2^-16 of a run's largest value (4e-5 measured); dense
    types and Q8_0 keep fp32 up to eight tokens (2e-7), everything else multiplies fp16 activations from two tokens on
    (4e-4 through q_a and q_b), as the MoE layers do ahead of the down projection (2.3e-4); prefill weights are fp16 too
    and pass through two products (5.7e-4)."""
    if case["kind"] in ("proj", "attn"):
        if case["t"] in DENSE + ("Q8_0",) and case["n"] <= 8:
            return {"rel": 1e-6}
        return {"rel": 1.6e-4 if case["n"] == 1 else 1.6e-3}
    if case["kind"] == "moe":
        return {"rel": 1e-3, "differ": 0.0}
    return {"rel": 2.4e-3, "differ": 0.0}


# ------------------------------------------------------------------------------------------------------------ inputs
def _buf(t, off=0, size=None):
    """A view of a tensor as the C ABI takes it."""
    total = t.numel() * t.element_size()
    return MsqBuffer(t.data_ptr(), off, total - off if size is None else size)


def _weights(t, n_elems, g):
    """Random blocks of one type, all finite: uniform payload bytes, fp16 scales of either format's usual size."""
    q = QType[t]
    if t in DENSE:
        w = torch.randn(n_elems, device=DEV, generator=g) * 0.02
        return w.to({"F32": torch.float32, "F16": torch.float16, "BF16": torch.bfloat16}[t]).view(torch.uint8)
    nb, bb = n_elems // block_elems(q), block_bytes(q)
    W = torch.randint(0, 256, (nb, bb), dtype=torch.uint8, device=DEV, generator=g)

    def half(sigma):
        return (torch.randn(nb, device=DEV, generator=g).abs() * sigma).to(torch.float16).view(torch.uint8).view(nb, 2)

    if t == "Q6_K":
        W[:, 208:210] = half(2e-5)
    else:
        W[:, 0:2] = half({"Q5_K": 5e-5, "Q8_0": 5e-4, "IQ4_NL": 5e-4, "IQ1_S": 0.004, "IQ2_XXS": 0.001}[t])
        if t == "Q5_K":
            W[:, 2:4] = half(5e-5)
    return W.view(-1)


def _out(*shape):
    return torch.zeros(shape, device=DEV)


def _check(rc):
    if rc:
        raise RuntimeError(_lib.load().msq_last_error().decode())


def _stream():
    return C.c_void_p(torch.cuda.current_stream().cuda_stream)


def prepare(case, seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    _check(_lib.load().msq_init())
    return {"proj": _prepare_proj, "attn": _prepare_attn, "moe": _prepare_moe, "prefill": _prepare_prefill}[case["kind"]](case, g)


def run(state):
    return state["run"](state)


# ----------------------------------------------------------------------------------------------- proj: one matrix a layer
def _prepare_proj(c, g):
    L, n, rows, cols = c["layers"], c["n"], c["rows"], c["cols"]
    nb = _row_bytes(c["t"], cols) * rows
    pitch = (nb + 255) // 256 * 256  # tensors of a model file start on aligned addresses
    W = torch.empty(L * pitch, dtype=torch.uint8, device=DEV)
    for i in range(L):
        W[i * pitch:i * pitch + nb] = _weights(c["t"], rows * cols, g)
    x = torch.randn(L, n, cols, device=DEV, generator=g)
    nw = 1 + 0.1 * torch.randn(cols, device=DEV, generator=g)
    xn, y = _out(n, cols), _out(L, n, rows)
    return {"run": _run_proj, "t": int(QType[c["t"]]), "rows": rows, "cols": cols, "n": n, "norm": c["norm"],
            "fused": n == 1 and c["t"] in NORM_FUSED and cols <= 12288, "keep": (W, x), "y": y, "xn": xn,
            "norm_w": _buf(nw), "nw": nw, "xnb": _buf(xn),
            "layers": [(_buf(W, i * pitch, nb), _buf(x[i]), _buf(y[i])) for i in range(L)]}


def _run_proj(s):
    L, st, t, rows, cols, n = _lib.load(), _stream(), s["t"], s["rows"], s["cols"], s["n"]
    nw, xn = C.byref(s["norm_w"]), C.byref(s["xnb"])
    for W, x, y in s["layers"]:
        if s["norm"] and s["fused"]:
            _check(L.msq_matvec_rmsnorm(st, t, C.byref(W), rows, cols, C.byref(x), nw, EPS, C.byref(y), 0))
            continue
        xin = C.byref(x)
        if s["norm"]:
            _check(L.msq_rmsnorm(st, C.byref(x), nw, xn, n, cols, EPS, 0, 0))
            xin = xn
        if n == 1:
            _check(L.msq_matvec(st, t, C.byref(W), rows, cols, xin, C.byref(y), 0, 1, None))
        else:
            _check(L.msq_matvec_n(st, t, C.byref(W), rows, cols, xin, C.byref(y), n, 0, 1))
    return s["y"]


# --------------------------------------------------------------------------------- attn: the projections of a layer
def _prepare_attn(c, g):
    L, n, t = c["layers"], c["n"], c["t"]
    shapes = _attn_shapes(c)
    layers, keep = [], []
    x = torch.randn(L, n, c["dim"], device=DEV, generator=g)
    att = torch.randn(L, n, c["heads"], device=DEV, generator=g)     # what attention hands to o_a
    mid = torch.randn(L, n, 8 * c["mid"], device=DEV, generator=g)   # ... and o_a to o_b
    nw = 1 + 0.1 * torch.randn(c["dim"], device=DEV, generator=g)
    outs = [_out(L, n, rows) for rows, _, _ in shapes]
    xn = _out(n, c["dim"])
    att16 = torch.zeros(n, c["heads"], dtype=torch.float16, device=DEV)
    for i in range(L):
        W = [_weights(t, rows * cols, g) for rows, cols, _ in shapes]
        keep.append(W)
        layers.append({"W": [_buf(w) for w in W], "x": _buf(x[i]), "att": _buf(att[i]), "mid": _buf(mid[i]), "y": [_buf(o[i]) for o in outs]})
    # o_a for many tokens: one strided product a group, group g's outputs behind those of group g - 1
    rows, cols, gr = shapes[3]
    wb, yb, r8 = _row_bytes(t, cols) * (rows // gr), 4 * n * (rows // gr), rows // gr
    for i, l in enumerate(layers):
        l["o_a"] = [(_buf(keep[i][3], k * wb, wb), _buf(att16, 2 * k * cols), _buf(outs[3][i], k * yb, yb)) for k in range(gr)]
    return {"run": _run_attn, "t": int(QType[t]), "n": n, "shapes": shapes, "layers": layers, "fused": n == 1 and t in NORM_FUSED, "keep": (keep, x, att, mid, att16, nw, xn),
            "norm_w": _buf(nw), "xn": _buf(xn), "att16": _buf(att16), "att_count": n * c["heads"], "heads": c["heads"], "r8": r8, "out": outs}


def _run_attn(s):
    L, st, t, n = _lib.load(), _stream(), s["t"], s["n"]
    (ra, ca, _), (rb, cb, _), (rk, ck, _), (ro, co, go), (rd, cd, _) = s["shapes"]
    nw, xn = C.byref(s["norm_w"]), C.byref(s["xn"])
    for l in s["layers"]:
        W, y = [C.byref(b) for b in l["W"]], [C.byref(b) for b in l["y"]]
        x = C.byref(l["x"])
        if s["fused"]:
            _check(L.msq_matvec_rmsnorm(st, t, W[0], ra, ca, x, nw, EPS, y[0], 0))
            _check(L.msq_matvec(st, t, W[1], rb, cb, y[0], y[1], 0, 1, None))
            _check(L.msq_matvec_rmsnorm(st, t, W[2], rk, ck, x, nw, EPS, y[2], 0))
            _check(L.msq_matvec(st, t, W[3], ro, co, C.byref(l["att"]), y[3], 0, go, None))
            _check(L.msq_matvec(st, t, W[4], rd, cd, C.byref(l["mid"]), y[4], 0, 1, None))
            continue
        _check(L.msq_rmsnorm(st, x, nw, xn, n, ca, EPS, 0, 0))
        if n <= 16:
            _check(L.msq_matvec_n(st, t, W[0], ra, ca, xn, y[0], n, 0, 1))
            _check(L.msq_matvec_n(st, t, W[1], rb, cb, y[0], y[1], n, 0, 1))
            _check(L.msq_matvec_n(st, t, W[2], rk, ck, xn, y[2], n, 0, 1))
            _check(L.msq_matvec_n(st, t, W[3], ro, co, C.byref(l["att"]), y[3], n, 0, go))
            _check(L.msq_matvec_n(st, t, W[4], rd, cd, C.byref(l["mid"]), y[4], n, 0, 1))
            continue
        _check(L.msq_matmul(st, t, W[0], ra, ca, xn, y[0], n, 0))
        _check(L.msq_matmul(st, t, W[1], rb, cb, y[0], y[1], n, 0))
        _check(L.msq_matmul(st, t, W[2], rk, ck, xn, y[2], n, 0))
        _check(L.msq_f32_to_f16(st, C.byref(l["att"]), C.byref(s["att16"]), s["att_count"]))
        for Wg, xg, yg in l["o_a"]:
            _check(L.msq_matmul_h(st, t, C.byref(Wg), s["r8"], co, C.byref(xg), C.byref(yg), n, 0, s["heads"]))
        _check(L.msq_matmul(st, t, W[4], rd, cd, C.byref(l["mid"]), y[4], n, 0))
    return s["out"]


# ------------------------------------------------------------------------------------- moe: one token, router and experts
def _expert_arena(c, g):
    """All experts of a layer in one allocation, gate | up | down behind each other; bytes of each."""
    gu, dn = _row_bytes(c["gu"], c["dim"]) * c["inter"], _row_bytes(c["dn"], c["inter"]) * c["dim"]
    per, E, n = 2 * gu + dn, c["experts"], c["dim"] * c["inter"]
    arena = torch.empty(E, per, dtype=torch.uint8, device=DEV)
    for e0 in range(0, E, 64):  # in parts, so that the generator's temporaries stay small
        arena[e0:e0 + 64, :2 * gu] = _weights(c["gu"], 64 * 2 * n, g).view(64, 2 * gu)
        arena[e0:e0 + 64, 2 * gu:] = _weights(c["dn"], 64 * n, g).view(64, dn)
    return arena, gu, dn


def _shared_expert(c, g):
    gu, dn = _row_bytes(c["sh"], c["dim"]) * c["inter"], _row_bytes(c["sh"], c["inter"]) * c["dim"]
    w = _weights(c["sh"], 3 * c["dim"] * c["inter"], g)
    return w, MsqExpertSlot(_buf(w, 0, gu), _buf(w, gu, gu), _buf(w, 2 * gu, dn))


def _prepare_moe(c, g):
    L, d, i, E = c["layers"], c["dim"], c["inter"], c["experts"]
    arena, gu, dn = _expert_arena(c, g)
    base, per = arena.data_ptr(), arena.shape[1]
    addr = base + per * torch.arange(E, device=DEV).view(E, 1) + torch.tensor([0, gu, 2 * gu], device=DEV).view(1, 3)
    router = (torch.randn(L, E, d, device=DEV, generator=g) * 0.02).to(torch.bfloat16)
    bias = 0.1 * torch.randn(E, device=DEV, generator=g)
    x = torch.randn(L, d, device=DEV, generator=g)
    y = torch.randn(L, d, device=DEV, generator=g)  # the residual stream: the layer's output is added to it
    ids = torch.zeros(L, TOPK, dtype=torch.int32, device=DEV)
    w = _out(L, TOPK)
    table = torch.zeros(L, TOPK, 3, dtype=torch.int64, device=DEV)
    h = torch.zeros(moe_decode_scratch_bytes(i), dtype=torch.uint8, device=DEV)
    rs = arch.Scratch.create(E)
    layers, keep = [], []
    for k in range(L):
        sw, slot = _shared_expert(c, g)
        keep.append(sw)
        a = MsqMoeDecodeArgs()
        a.t_gate_up, a.t_down, a.t_shared, a.n_routed, a.has_shared = int(QType[c["gu"]]), int(QType[c["dn"]]), int(QType[c["sh"]]), TOPK, 1
        a.shared, a.weights, a.x, a.y, a.scratch, a.dim, a.inter = slot, _buf(w[k]), _buf(x[k]), _buf(y[k]), _buf(h), d, i
        layers.append({"args": a, "x": _buf(x[k]), "W": _buf(router[k]), "ids_t": ids[k], "ids": _buf(ids[k]), "w": _buf(w[k]), "table_t": table[k], "table": _buf(table[k])})
    return {"run": _run_moe, "dim": d, "experts": E, "addr": addr, "layers": layers, "keep": (arena, router, bias, x, h, rs, keep), "bias": _buf(bias),
            "scratch": _buf(rs.mem), "ids": ids, "w": w, "y": y}


def _run_moe(s):
    L, st = _lib.load(), _stream()
    bias, scratch, bf16 = C.byref(s["bias"]), C.byref(s["scratch"]), int(QType.BF16)
    for l in s["layers"]:
        _check(L.msq_router_fused(st, bf16, C.byref(l["x"]), C.byref(l["W"]), bias, scratch, C.byref(l["ids"]), C.byref(l["w"]), s["dim"], s["experts"], arch.ROUTE_SCALE))
        torch.index_select(s["addr"], 0, l["ids_t"], out=l["table_t"])
        _check(L.msq_moe_decode_table(st, C.byref(l["args"]), C.byref(l["table"])))
    return {"y": s["y"], "ids": s["ids"], "w": s["w"]}


# ------------------------------------------------------------------------------ prefill: routing and the grouped GEMMs
def _prepare_prefill(c, g):
    n, d, i, E = c["n"], c["dim"], c["inter"], c["experts"]
    arena, gu, dn = _expert_arena(c, g)
    # logits whose top-6 are draws from a Zipf popularity over the experts (Gumbel noise: sampling without replacement)
    u = torch.rand(n, E, device=DEV, generator=g).clamp(1e-9, 1 - 1e-7)
    rank = torch.randperm(E, device=DEV, generator=g)
    logits = (-c["zipf"] * torch.log(rank + 1.0) - torch.log(-torch.log(u))).contiguous()
    bias = torch.zeros(E, device=DEV)
    ids = torch.zeros(n, TOPK, dtype=torch.int32, device=DEV)
    w = _out(n, TOPK)
    x = torch.randn(n, d, device=DEV, generator=g)
    x = x.to(torch.bfloat16) if c["bf16"] else x
    y = torch.randn(n, d, device=DEV, generator=g)
    lists = arch.RouteLists.create(n, E)
    s = {"run": _run_prefill, "n": n, "experts": E, "logits": _buf(logits), "bias": _buf(bias), "ids": _buf(ids), "w": _buf(w), "lists": lists.c(), "y": y, "ids_t": ids, "w_t": w}
    L, st = _lib.load(), _stream()
    _check(L.msq_router_topk(st, C.byref(s["logits"]), C.byref(s["bias"]), C.byref(s["ids"]), C.byref(s["w"]), n, E, arch.ROUTE_SCALE))
    _check(L.msq_route_lists(st, C.byref(s["ids"]), C.byref(s["w"]), n, E, C.byref(s["lists"])))
    offs = lists.t_offsets.cpu().tolist()  # the grouped GEMM takes the offsets from the host
    used = [e for e in range(E) if offs[e + 1] > offs[e]]
    slots = (MsqExpertSlot * len(used))(*[MsqExpertSlot(_buf(arena[e], 0, gu), _buf(arena[e], gu, gu), _buf(arena[e], 2 * gu, dn)) for e in used])
    host_offs = (C.c_int * (len(used) + 1))(*([offs[e] for e in used] + [offs[E]]))
    a = MsqMoePrefillArgs()
    a.t_gate_up, a.t_down, a.n_tokens, a.n_exp, a.slots, a.offs = int(QType[c["gu"]]), int(QType[c["dn"]]), n, len(used), slots, host_offs
    a.tok, a.wt, a.slot_of, a.k_per_token = lists.tok.c(), lists.w.c(), lists.slot_of.c(), TOPK
    keep = [arena, logits, bias, x, lists, slots, host_offs]
    if c["sh"]:
        sw, slot = _shared_expert(c, g)
        keep.append(sw)
        a.has_shared, a.t_shared, a.shared = 1, int(QType[c["sh"]]), slot
    scratch = torch.empty(moe_prefill_scratch_bytes(n * TOPK, n, len(used), d, i), dtype=torch.uint8, device=DEV)
    a.X, a.Y, a.scratch, a.path, a.shared_dense, a.dim, a.inter, a.x_is_bf16 = _buf(x), _buf(y), _buf(scratch), -1, -1, d, i, int(c["bf16"])
    keep.append(scratch)
    s.update(args=a, keep=keep)
    return s


def _run_prefill(s):
    L, st = _lib.load(), _stream()
    _check(L.msq_router_topk(st, C.byref(s["logits"]), C.byref(s["bias"]), C.byref(s["ids"]), C.byref(s["w"]), s["n"], s["experts"], arch.ROUTE_SCALE))
    _check(L.msq_route_lists(st, C.byref(s["ids"]), C.byref(s["w"]), s["n"], s["experts"], C.byref(s["lists"])))
    _check(L.msq_moe_prefill(st, C.byref(s["args"])))
    return {"y": s["y"], "ids": s["ids_t"], "w": s["w_t"]}
