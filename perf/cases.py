"""What this library is timed on: blocks of one FastConformer encoder layer,
single quantized linears, the joint GEMV and the greedy TDT decode, each
called through the package's entry points as a host program calls them.

Sizes are the model's own (width 1024, feed-forward 4096, convolution 2048, 8
heads of 128, joint 640 -> 1025 tokens + 5 durations); frames run from a short
utterance to one hour of audio at 80 ms a frame (45000).
"""
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "l4-parakeet-rs_amd"))

import parakeet_linear as pk  # noqa: E402

D, FF, CONV, HEADS, HEAD, POS, LEFT = 1024, 4096, 2048, 8, 128, 272, 128
H, TOKENS, DURATIONS = 640, 1025, 5
EPS = 1e-5
FP8_INPUT_SCALE = 8.0 / 448.0
LONG_ROWS = 1040   # padded frames from which a layer takes the long-form plan
SHORT_ROWS = 512   # below this the attention is the fp16 short form
MOST_FRAMES, MOST_DECODE = 45000, 7500


def listed():
    return [
        # First half of a layer (norm pair, FF1, norm, QKV): a 7.4 s utterance, one
        # hour of audio in one request.
        {"name": "front_clip", "kind": "front", "rows": 93},
        {"name": "front_hour", "kind": "front", "rows": 45000},
        # Attention with its packers and the output projection: one minute (fp16
        # scores), one hour (packed INT4 / INT8).
        {"name": "attend_minute", "kind": "attend", "rows": 750},
        {"name": "attend_hour", "kind": "attend", "rows": 45000},
        # Second half of a layer (convolution pointwise linears, FF2, norm pair): one
        # minute (FP8 FF2), 26 minutes less a ragged end (INT4 x INT4 with 2:4 sparse contract).
        {"name": "tail_minute", "kind": "tail", "rows": 750},
        {"name": "tail_long", "kind": "tail", "rows": 20011},
        # Single linears on fp16 activations, quantizing them per row where the format asks for it:
        # INT8 with fp32 output for one minute, INT4-g128 on INT8 activations for a
        # ten-minute file, INT4-g128 on fp16 activations at a ragged half hour.
        {"name": "int8_minute", "kind": "linear", "format": "int8", "m": 750, "n": 4096, "k": 1024, "fp32": True},
        {"name": "g128_int8_10min", "kind": "linear", "format": "g128_int8", "m": 7500, "n": 1024, "k": 4096, "fp32": False},
        {"name": "g128_fp16_long", "kind": "linear", "format": "g128_fp16", "m": 22111, "n": 4096, "k": 1024, "fp32": False},
        # One joint step of a host-driven greedy loop: the smallest call.
        {"name": "joint_step", "kind": "joint", "steps": 1, "int8": True},
        # Whole greedy decode of one utterance after the encoder: 7.4 s (fp16
        # prediction network), ten minutes (INT8 recurrence and input table).
        {"name": "decode_clip", "kind": "decode", "frames": 93, "int8": True},
        {"name": "decode_10min", "kind": "decode", "frames": 7500, "int8": True},
    ]


def _log(rng, lo, hi):
    return min(hi, int(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["front", "front", "attend", "attend", "tail", "tail", "linear", "linear", "linear", "joint", "decode", "decode"])
    if kind in ("front", "attend", "tail"):
        return {"kind": kind, "rows": _log(rng, 17, MOST_FRAMES)}
    if kind == "linear":
        n, k = rng.choice([(3072, 1024), (1024, 1024), (4096, 1024), (1024, 4096), (2048, 1024), (640, 1024)])
        return {"kind": kind, "format": rng.choice(["int8", "fp8", "g128_int8", "g128_fp16", "fp16"]),
                "m": _log(rng, 11, MOST_FRAMES // 2 if k > 1024 else MOST_FRAMES), "n": n, "k": k, "fp32": rng.random() < 0.25}
    if kind == "joint":
        return {"kind": kind, "steps": _log(rng, 1, 4096), "int8": rng.random() < 0.7}
    return {"kind": kind, "frames": _log(rng, 20, MOST_DECODE), "int8": rng.random() < 0.8}


# ---- inputs -----------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, *shape, scale=1.0):
    return (torch.randn(shape, generator=g, device="cuda") * scale).half()


def _u8(*shape):
    return torch.empty(shape, dtype=torch.uint8, device="cuda")


def _f16(*shape):
    return torch.zeros(shape, dtype=torch.float16, device="cuda")


def _f32(*shape):
    return torch.empty(shape, dtype=torch.float32, device="cuda")


def _padded(rows):
    return (rows + 15) // 16 * 16


def _norm(g):
    return (torch.rand(D, generator=g, device="cuda") + 0.5).half(), _randn(g, D, scale=0.1)


def _frames(g, rows, padded, scale=2.0):
    x = _randn(g, padded, D, scale=scale)
    x[rows:] = 0
    return x


def _raw(case, seed):
    """The fp16 / fp32 tensors of a case: what the model file and the previous
    stage hand over, before anything is packed."""
    g = _gen(seed)
    kind = case["kind"]
    s = {}
    if kind in ("front", "attend", "tail"):
        rows, padded = case["rows"], _padded(case["rows"])
        s["x"] = _frames(g, rows, padded)
    if kind == "front":
        s.update(n1=_norm(g), n2=_norm(g), n3=_norm(g), up=_randn(g, FF, D, scale=0.02), down=_randn(g, D, FF, scale=0.02),
                 qkv=_randn(g, 3 * D, D, scale=0.02))
    elif kind == "attend":
        s.update(q=_frames(g, rows, padded, 1.0), k=_frames(g, rows, padded, 1.0), v=_frames(g, rows, padded, 1.0),
                 pos=_randn(g, HEADS * POS, HEAD), bu=_randn(g, D, scale=0.1), bv=_randn(g, D, scale=0.1),
                 o=_randn(g, D, D, scale=0.02))
    elif kind == "tail":
        s.update(n1=_norm(g), n2=_norm(g), n3=_norm(g), n4=_norm(g), pw1=_randn(g, CONV, D, scale=0.05),
                 pw2=_randn(g, D, D, scale=0.02), up=_randn(g, FF, D, scale=0.02), down=_randn(g, D, FF, scale=0.02))
    elif kind == "linear":
        s.update(x=_randn(g, case["m"], case["k"]), w=_randn(g, case["n"], case["k"], scale=0.02),
                 bias=torch.randn(case["n"], generator=g, device="cuda") * 0.1)
    else:
        r = lambda *shape, scale: torch.randn(shape, generator=g, device="cuda") * scale  # noqa: E731
        s.update(joint=_randn(g, TOKENS + DURATIONS, H, scale=0.08), joint_bias=r(TOKENS + DURATIONS, scale=0.1))
        # blank favoured, duration 1 preferred and 0 rare: a token about every five frames, as in speech
        s["joint_bias"][TOKENS - 1] += 2.3
        s["joint_bias"][TOKENS] -= 3.0
        s["joint_bias"][TOKENS + 1] += 0.5
        if kind == "joint":
            s.update(enc=_randn(g, case["steps"], H, scale=0.5), pred=r(H, scale=0.5))
        else:
            s["enc"] = _randn(g, case["frames"], H, scale=0.5)
            s["emb"] = _randn(g, TOKENS - 1, H, scale=0.5)
            s["lstm"] = [f for _ in range(2) for f in (_randn(g, 4 * H, H, scale=0.05), _randn(g, 4 * H, H, scale=0.05),
                                                       r(4 * H, scale=0.1), r(4 * H, scale=0.1))]
            s["proj"] = (_randn(g, H, H, scale=0.1), r(H, scale=0.1))
    return s


def _pack_fp8(w):
    n, k = w.shape
    q, s = _u8(n, k), _f32(n)
    pk.call("pk_pack_fp8_rows", w, n, k, q, s)
    return q, s


def prepare(case, seed):
    """Weights packed as the loader packs them, inputs on the GPU, and the
    buffers a program keeps for its activations."""
    s = _raw(case, seed)
    kind = case["kind"]
    s["case"] = dict(case)
    if kind in ("front", "attend", "tail"):
        p = _padded(case["rows"])
        s.update(rows=case["rows"], p=p, state=_f16(p, D), x8=_u8(p, D), xs=_f32(p))
    if kind == "front":
        for name in ("up", "down", "qkv"):
            s[name] = _pack_fp8(s[name])
        s.update(h8=_u8(p, FF), out=_f16(p, 3 * D))
    elif kind == "attend":
        s["o"] = _pack_fp8(s["o"])
        if p < SHORT_ROWS:
            s["ctx"] = _f16(p, D)
        else:
            s["v"] = s["v"].t().contiguous()
            s["value"] = _u8(p * D + p * D // 2 + 4096)
            s["ctx"] = _u8(p, D) if p >= LONG_ROWS else _f16(p, D)
            if p >= LONG_ROWS:
                s["packed"] = {"key": _u8(p * 512), "key_scales": _f32(p * 8), "position": _u8(HEADS * POS * HEAD),
                               "position_scales": _f32(HEADS * POS)}
    elif kind == "tail":
        for name in ("pw1", "pw2", "down"):
            s[name] = _pack_fp8(s[name])
        s.update(glu=_f16(p, D), out=_f16(p, D), next8=_u8(p, D))
        if p >= LONG_ROWS:
            n4, ns, n6 = _u8(FF, D // 2), _f32(FF), _u8(FF, D)
            pk.call("pk_pack_int4_rows", s["up"], FF, D, n4, ns)
            pk.call("pk_unpack_int4_fp6", n4, n6, FF * D)
            s.update(up=(n6, ns), h8=_u8(p * (FF // 2 + FF // 8)))
        else:
            s.update(up=_pack_fp8(s["up"]), h8=_u8(p, FF))
    elif kind == "linear":
        m, n, k, fmt = case["m"], case["n"], case["k"], case["format"]
        s["out"] = _f32(m, n) if case["fp32"] and fmt != "fp16" else _f16(m, n)
        if fmt in ("int8", "g128_int8"):
            s.update(x8=torch.empty((m, k), dtype=torch.int8, device="cuda"), xs=_f32(m))
        if fmt == "fp8":
            s.update(x8=_u8(m, k), xs=_f32(m), w=_pack_fp8(s["w"]))
        elif fmt == "int8":
            q, ws = torch.empty((n, k), dtype=torch.int8, device="cuda"), _f32(n)
            pk.call("pk_pack_int8_rows", s["w"], n, k, q, ws)
            s["w"] = (q, ws)
        elif fmt.startswith("g128"):
            q = torch.empty((n, k // 8), dtype=torch.int32, device="cuda")
            gs, gz = _f16(n, k // 128), _f16(n, k // 128)
            pk.call("pk_pack_int4_g128", s["w"], n, k, q, gs, gz)
            s["w"] = (q, gs, gz)
    else:
        w = s["joint"]
        s["joint_scales"] = None
        if case["int8"]:
            q, ws = torch.empty(w.shape, dtype=torch.int8, device="cuda"), _f32(w.shape[0])
            pk.call("pk_pack_int8_rows", w, w.shape[0], H, q, ws)
            s.update(joint=q, joint_scales=ws)
        if kind == "joint":
            s.update(scores=_f32(case["steps"], TOKENS + DURATIONS),
                     decision=torch.zeros((case["steps"], 2), dtype=torch.int32, device="cuda"))
        else:
            words = pk.lib.pk_tdt_decode_workspace_bytes(H) // 4
            s.update(tokens=torch.zeros(case["frames"] * 10, dtype=torch.int32, device="cuda"),
                     result=torch.zeros(4, dtype=torch.int32, device="cuda"),
                     workspace=torch.empty(words, dtype=torch.int32, device="cuda"),
                     table=_f16(TOKENS - 1, 4 * H) if case["frames"] >= pk.LONG_DECODE_MIN_FRAMES else None)
    return s


# ---- one pass ----------------------------------------------------------------------

def _front(s):
    p, rows = s["p"], s["rows"]
    pk.call("pk_layer_norm_pair", s["x"], *s["n1"], s["state"], *s["n2"], s["x8"], rows, p, EPS, 1.0 / FP8_INPUT_SCALE)
    pk.call("pk_ffn_expand_fp8_packed", s["x8"], *s["up"], None, s["h8"], p, FP8_INPUT_SCALE, 0)
    pk.call("pk_ffn_contract_fp8", s["h8"], *s["down"], s["state"], p)
    pk.call("pk_layer_norm_quantize_fp8_dynamic", s["state"], *s["n3"], s["x8"], s["xs"], rows, p, EPS)
    pk.call("pk_linear_fp8_dyn", s["x8"], s["xs"], *s["qkv"], None, s["out"], 0, p, 3 * D, D)
    return {"state": s["state"], "qkv": s["out"]}


def _attend(s):
    p, rows = s["p"], s["rows"]
    w, ws = s["o"]
    if p < SHORT_ROWS:
        pk.launch_attention_arena(s["q"], s["k"], None, s["pos"], s["bu"], s["bv"], s["ctx"], rows, p, rows, p, value=s["v"])
    elif p < LONG_ROWS:
        pk.call("pk_quantize_value_int4", s["v"], s["value"], p * D, 56.0)
        pk.launch_attention_arena(s["q"], s["k"], s["value"], s["pos"], s["bu"], s["bv"], s["ctx"], rows, p, rows, p)
    else:
        pk.call("pk_quantize_value_int4_register", s["v"], s["value"], p * D, 56.0, rows)
        pk.launch_attention_arena(s["q"], s["k"], s["value"], s["pos"], s["bu"], s["bv"], s["ctx"], rows, p, rows, p,
                                  packed=s["packed"])
        pk.gemm(pk.FMT_FP8, pk.EPI_F16, s["ctx"], w, p, D, D, s["state"], w_scales=ws, in_scale=1.0 / 28.0, residual=s["x"],
                res_scale=1.0)
        return {"context": s["ctx"].view(torch.float8_e4m3fn), "state": s["state"]}
    pk.call("pk_quantize_rows1024", s["ctx"], s["x8"], s["xs"], p)
    pk.gemm(pk.FMT_FP8, pk.EPI_F16, s["x8"], w, p, D, D, s["state"], w_scales=ws, row_scales=s["xs"], residual=s["x"], res_scale=1.0)
    return {"context": s["ctx"], "state": s["state"]}


def _tail(s):
    p, rows = s["p"], s["rows"]
    pk.call("pk_layer_norm_quantize_fp8_dynamic", s["x"], *s["n1"], s["x8"], s["xs"], rows, p, EPS)
    pk.call("pk_conv_glu_fp8", s["x8"], *s["pw1"], s["xs"], s["glu"], p, rows)
    pk.call("pk_quantize_rows1024", s["glu"], s["x8"], s["xs"], p)
    pk.gemm(pk.FMT_FP8, pk.EPI_F16, s["x8"], s["pw2"][0], p, D, D, s["state"], w_scales=s["pw2"][1], row_scales=s["xs"],
            residual=s["x"], res_scale=1.0)
    if p >= LONG_ROWS:
        pk.call("pk_layer_norm_quantize_int4_fp6", s["state"], *s["n2"], s["x8"], s["xs"], rows, p, EPS)
        pk.call("pk_ffn_expand_int4_sparse_fp6", s["x8"], *s["up"], s["xs"], s["h8"], p, 1.0, 1)
        pk.call("pk_ffn_contract_fp8_sparse", s["h8"], *s["down"], s["state"], p, FF)
    else:
        pk.call("pk_layer_norm_quantize_fp8_dynamic", s["state"], *s["n2"], s["x8"], s["xs"], rows, p, EPS)
        pk.call("pk_ffn_expand_fp8_packed", s["x8"], *s["up"], s["xs"], s["h8"], p, 1.0, 1)
        pk.call("pk_ffn_contract_fp8", s["h8"], *s["down"], s["state"], p)
    pk.call("pk_layer_norm_pair", s["state"], *s["n3"], s["out"], *s["n4"], s["next8"], rows, p, EPS, 1.0 / FP8_INPUT_SCALE)
    return {"glu": s["glu"], "state": s["state"], "out": s["out"], "next": s["next8"].view(torch.float8_e4m3fn)}


def _linear(s):
    c = s["case"]
    m, n, k, fmt, f32 = c["m"], c["n"], c["k"], c["format"], int(s["out"].dtype == torch.float32)
    if fmt == "fp16":
        pk.launch_linear(s["x"], s["w"], s["bias"], None, s["out"], m, n, k)
    elif fmt == "g128_fp16":
        pk.call("pk_linear_int4g128", s["x"], *s["w"], s["bias"], s["out"], f32, m, n, k)
    else:
        pk.call("pk_quantize_rows", 0 if fmt == "fp8" else 1, s["x"], s["x8"], s["xs"], m, m, k)
        entry = {"fp8": "pk_linear_fp8_dyn", "int8": "pk_linear_int8_dyn", "g128_int8": "pk_linear_int4g128_a8"}[fmt]
        pk.call(entry, s["x8"], s["xs"], *s["w"], s["bias"], s["out"], f32, m, n, k)
    return s["out"]


def _joint(s):
    c = s["case"]
    pk.call("pk_joint_gemv", s["joint"], int(c["int8"]), s["joint_scales"], s["joint_bias"], s["enc"], s["pred"], s["scores"],
            s["decision"], TOKENS + DURATIONS, H, TOKENS, DURATIONS, c["steps"], H)
    return {"scores": s["scores"], "decision": s["decision"]}


def _decode(s):
    c = s["case"]
    pk.launch_decode(s["enc"], c["frames"], [s["emb"], *s["lstm"]], s["proj"], (s["joint"], s["joint_bias"]), s["tokens"],
                     s["result"], s["workspace"], input_table=s["table"], joint_int8=c["int8"], joint_scales=s["joint_scales"],
                     hidden=H, token_outputs=TOKENS, durations=DURATIONS)
    out = {"tokens": s["tokens"], "result": s["result"]}
    if s["table"] is not None:
        out["table"] = s["table"]
    return out


def run(state):
    return {"front": _front, "attend": _attend, "tail": _tail, "linear": _linear, "joint": _joint,
            "decode": _decode}[state["case"]["kind"]](state)


# ---- what a pass cannot do without -----------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind in ("front", "attend", "tail"):
        r = _padded(case["rows"])
        if kind == "front":
            w = FF * D * 2 + 3 * D * D
            return {"bytes": r * 2 * (D + D + 3 * D) + w, "flops": 2 * r * w}
        if kind == "tail":
            w = CONV * D + D * D + 2 * FF * D
            return {"bytes": r * (2 * D * 4 + D) + w, "flops": 2 * r * w}
        span = min(r, 2 * LEFT + 1)
        return {"bytes": r * 2 * D * 5 + r * D * (1 if r >= LONG_ROWS else 2) + HEADS * POS * HEAD * 2 + D * D,
                "flops": 2 * r * (D * D + 3 * span * D)}
    if kind == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        wb = {"fp16": 2.0, "int8": 1.0, "fp8": 1.0}.get(case["format"], 0.53)
        return {"bytes": m * k * 2 + n * k * wb + m * n * (4 if case["fp32"] and case["format"] != "fp16" else 2), "flops": 2.0 * m * n * k}
    outs = TOKENS + DURATIONS
    if kind == "joint":
        return {"bytes": outs * H * (1 if case["int8"] else 2) + case["steps"] * (H * 2 + outs * 4 + 8), "flops": 2 * case["steps"] * outs * H}
    # one joint per frame, one prediction update per token (about every fifth frame)
    t = case["frames"]
    w = 4 * H * H * 4 + H * H
    table = 2 * (TOKENS - 1) * 4 * H * H if t >= pk.LONG_DECODE_MIN_FRAMES else 0
    return {"bytes": t * H * 2 + 2 * w + outs * H * (1 if case["int8"] else 2) + (TOKENS - 1) * H * 2,
            "flops": 2 * t * outs * H + 2 * (t // 5) * w + table}


def tolerance(case):
    """About four times what a pass is from exact(): a sum in another order moves
    fp32 results in the last places, fp16 ones by a rounding, and in the chains
    some roundings of the 8-bit intermediates then fall the other way (a norm's
    e4m3 output after a chain is 0.009 off).  Joint and decode decisions are whole numbers."""
    kind = case["kind"]
    if kind == "decode":
        return "exact"
    if kind == "joint":
        return {"rel": 1e-6, "max": 1e-5}
    if kind == "linear":
        fine = case["fp32"] and case["format"] in ("int8", "fp8", "g128_int8")
        return {"rel": 1e-5, "max": 1e-4} if fine else {"rel": 1e-3, "max": 1e-2}
    return {"rel": 2e-2, "max": 0.5}


# ---- the same in 64 bits ------------------------------------------------------------

def _round_to(x, bits, least):
    """x to `bits` stored mantissa bits, ties to even; exponents below `least` are subnormal."""
    _, e = torch.frexp(x)
    step = torch.exp2((e - 1).clamp(min=least).double() - bits)
    return torch.round(x / step) * step


def _e4m3(x):
    return _round_to(x.clamp(-448.0, 448.0), 3, -6)


def _half(x):
    return _round_to(x, 10, -14)


def _over(x, c):
    """fp32 x / c correctly rounded (by a Python number, torch multiplies with 1 / c)."""
    return x / torch.full((1,), float(c), device="cuda")


def _rows_fp8(x):
    """Per-row dynamic e4m3: (codes, scale), scale and quotient in fp32 as stored."""
    x = x.float()
    s = _over(x.abs().amax(1, keepdim=True), 448)
    s = torch.where(s > 0, s, torch.ones_like(s))
    return _e4m3((x / s).double()), s.double()


def _ints(x, s, lo, hi):
    return torch.round(x.float() / s).clamp(lo, hi).double()


def _dequant(w):
    q, s = _rows_fp8(w)
    return q * s


def _ln(x, n):
    x = x.double()
    y = (x - x.mean(1, keepdim=True)) / torch.sqrt(x.var(1, unbiased=False, keepdim=True) + EPS)
    return _half(y * n[0].double() + n[1].double())


def _ff_hidden(v):
    return _e4m3(_half(v * torch.sigmoid(v)) * 16.0)


def _ln8(x, n):
    q, s = _rows_fp8(_ln(x, n))
    return q * s


def _chunks(rows, step=7504):
    return [slice(a, min(rows, a + step)) for a in range(0, rows, step)]


def _exact_front(s, case):
    rows, p = case["rows"], _padded(case["rows"])
    state = torch.zeros((p, D), dtype=torch.float64, device="cuda")
    qkv = torch.zeros((p, 3 * D), dtype=torch.float64, device="cuda")
    up, down, wq = _dequant(s["up"]), _dequant(s["down"]), _dequant(s["qkv"])
    for c in _chunks(rows):
        y = _ln(s["x"][c], s["n1"])
        x8 = _e4m3(_ln(y, s["n2"]) / FP8_INPUT_SCALE) * FP8_INPUT_SCALE
        state[c] = _half(y + 0.5 * (_ff_hidden(x8 @ up.t()) / 16.0 @ down.t()))
        qkv[c] = _ln8(state[c], s["n3"]) @ wq.t()
    return {"state": state, "qkv": qkv}


def _top2(h):
    """The two largest magnitudes of every quartet, ties to the lower index."""
    q = h.reshape(h.shape[0], -1, 4)
    a = q.abs()
    keep = torch.zeros_like(q)
    for i in range(4):
        beaten = sum(((a[..., j] > a[..., i]) | ((a[..., j] == a[..., i]) & (j < i))).int() for j in range(4) if j != i)
        keep[..., i] = (beaten < 2).double()
    return (q * keep).reshape(h.shape)


def _exact_tail(s, case):
    rows, p = case["rows"], _padded(case["rows"])
    r = {n: torch.zeros((p, D), dtype=torch.float64, device="cuda") for n in ("glu", "state", "out", "next")}
    pw1, pw2, down = _dequant(s["pw1"]), _dequant(s["pw2"]), _dequant(s["down"])
    if p >= LONG_ROWS:
        w = s["up"].float()
        ws = torch.maximum(_over(w, 7), _over(-w, 8)).amax(1, keepdim=True)
        up = _ints(w, ws, -8, 7) * ws.double()
    else:
        up = _dequant(s["up"])
    for c in _chunks(rows):
        v = _half(_ln8(s["x"][c], s["n1"]) @ pw1.t())
        r["glu"][c] = _half(v[:, :D] * torch.sigmoid(v[:, D:]))
        q, qs = _rows_fp8(r["glu"][c])
        y = _half(s["x"][c].double() + (q * qs) @ pw2.t())
        if p >= LONG_ROWS:
            n = _ln(y, s["n2"]).float()
            ns = torch.maximum(_over(n, 7), _over(-n, 8)).amax(1, keepdim=True)
            hidden = _top2(_ff_hidden((_ints(n, ns, -8, 7) * ns.double()) @ up.t()))
        else:
            hidden = _ff_hidden(_ln8(y, s["n2"]) @ up.t())
        y = _half(y + 0.5 * (hidden / 16.0 @ down.t()))
        r["state"][c] = y
        r["out"][c] = _ln(y, s["n3"])
        r["next"][c] = _e4m3(_ln(r["out"][c], s["n4"]) / FP8_INPUT_SCALE)
    return r


def _windows(x, lo, hi):
    """Rows lo .. hi - 1 of x, zeros where there are none."""
    out = torch.zeros((hi - lo, x.shape[1]), dtype=torch.float64, device="cuda")
    a, b = max(lo, 0), min(hi, x.shape[0])
    out[a - lo:b - lo] = x[a:b].double()
    return out


def _attention(q, k, v, pos, bu, bv, rows, first, last, bf16_scores=False, u4=False):
    """Queries first .. last - 1 of plain local relative-position attention on
    [8 heads x rows x 128] operands; with u4 the probabilities in fifteenths."""
    n = last - first
    out = torch.zeros((n, D), dtype=torch.float64, device="cuda")
    rel = torch.arange(2 * LEFT + 1, device="cuda")
    at = torch.arange(n, device="cuda")[:, None] + rel[None]          # key column of (query, slot)
    key = at + first - LEFT
    seen = (key >= 0) & (key < rows)
    for h in range(HEADS):
        c = slice(h * HEAD, (h + 1) * HEAD)
        kw, vw = _windows(k[:, c], first - LEFT, last + LEFT), _windows(v[:, c], first - LEFT, last + LEFT)
        content = (q[0][first:last, c] @ kw.t()).gather(1, at)
        place = q[1][first:last, c] @ pos[h][: 2 * LEFT + 1].double().t()
        if bf16_scores:
            content, place = _round_to(content, 7, -126), _round_to(place, 7, -126)
        e = ((content + place) / HEAD ** 0.5).masked_fill(~seen, float("-inf"))
        e = torch.exp(e - e.amax(1, keepdim=True))
        den = e.sum(1, keepdim=True)
        w = torch.round(e * 15.0) / (15.0 * den) if u4 else e / den
        out[:, c] = torch.zeros((n, kw.shape[0]), dtype=torch.float64, device="cuda").scatter_(1, at, w) @ vw
    return out


def _exact_attend(s, case):
    rows, p = case["rows"], _padded(case["rows"])
    pos = s["pos"].reshape(HEADS, POS, HEAD)
    ctx = torch.zeros((p, D), dtype=torch.float64, device="cuda")
    q = s["q"].double()
    qb = (q + s["bu"].double(), q + s["bv"].double())
    edge = min(rows, 272)
    if p < LONG_ROWS:
        v = s["v"].double() if p < SHORT_ROWS else _e4m3(s["v"].double() * 56.0) / 56.0
        for a in range(0, rows, 1024):
            ctx[a:min(rows, a + 1024)] = _attention(qb, s["k"], v, pos, None, None, rows, a, min(rows, a + 1024))
        ctx = _half(ctx)
        c8, cs = _rows_fp8(ctx)
        y = c8 * cs
    else:
        def ints(x, top):  # per-vector symmetric codes times their scale
            x = x.float()
            sc = _over(x.abs().amax(-1, keepdim=True), top)
            sc = torch.where(sc > 0, sc, torch.ones_like(sc))
            return _ints(x, sc, -top, top) * sc.double()

        heads = lambda x, top: ints(x.reshape(p, HEADS, HEAD), top).reshape(p, D)  # noqa: E731
        qq = (heads(_half(qb[0]), 7), heads(_half(qb[1]), 127))
        k4, p8, v4 = heads(s["k"], 7), ints(pos, 127), ints(s["v"].t(), 7).t()
        for a in range(0, rows, 1024):
            b = min(rows, a + 1024)
            ctx[a:b] = _attention(qq, k4, v4, p8, None, None, rows, a, b, True, True)
        # queries whose 16-row tile has keys outside [0, rows): fp16 operands, e4m3 values
        v8 = _e4m3(s["v"].double() * 56.0) / 56.0
        tiles = [t for t in range(0, p, 16) if t < LEFT or t + 15 + LEFT >= rows]
        for a, b in ((0, LEFT), (next(t for t in tiles if t > LEFT), rows)):
            ctx[a:b] = _attention(qb, s["k"], v8, pos, None, None, rows, a, b)
        ctx = _e4m3(_half(ctx) * 28.0)
        y = ctx / 28.0
    state = torch.zeros((p, D), dtype=torch.float64, device="cuda")
    state[:] = s["x"].double() + y @ _dequant(s["o"]).t()
    return {"context": ctx, "state": state}


def _exact_linear(s, case):
    x, w, fmt = s["x"], s["w"], case["format"]

    def int8(a):
        sc = _over(a.float().abs().amax(1, keepdim=True), 127)
        return _ints(a, sc, -127, 127) * sc.double()

    if fmt.startswith("g128"):
        g = w.float().reshape(case["n"], -1, 128)
        lo, hi = g.amin(2, keepdim=True).clamp(max=0), g.amax(2, keepdim=True).clamp(min=0)
        sc = _over(hi - lo, 15).half().float()
        sc = torch.where(sc > 0, sc, torch.ones_like(sc))
        z = torch.round(-lo / sc).clamp(0, 15)
        q = (torch.round(g / sc).clamp(-64, 64) + z).clamp(0, 15) - z
        w = (q.double() * sc.double()).reshape(case["n"], case["k"])
    else:
        w = {"fp8": _dequant, "int8": int8, "fp16": torch.Tensor.double}[fmt](w)
    x = _dequant(x) if fmt == "fp8" else int8(x) if fmt in ("int8", "g128_int8") else x.double()
    return x @ w.t() + s["bias"].double()


def _joint_scores(s, case, enc, pred):
    w = s["joint"]
    if case["int8"]:
        sc = _over(w.float().abs().amax(1, keepdim=True), 127)
        w = _ints(w, sc, -127, 127) * sc.double()
    return (enc.double() + pred.double()).clamp(min=0) @ w.double().t() + s["joint_bias"].double()


def exact(case, seed):
    kind = case["kind"]
    if kind == "decode":
        return None  # every decision feeds the next: no value in 64 bits stands for it
    s = _raw(case, seed)
    if kind == "joint":
        return {"scores": _joint_scores(s, case, s["enc"], s["pred"]), "decision": None}
    return {"front": _exact_front, "attend": _exact_attend, "tail": _exact_tail, "linear": _exact_linear}[kind](s, case)
