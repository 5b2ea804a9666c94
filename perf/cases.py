"""What programs that use thq have it do, as cases that can be timed and checked.

A case is one call, or the few calls of one block of a decoder, through the
package's public entry points: a projection, the MLP (gate/up + down), a whole
decoder layer's four projections, or the LM head with its greedy or sampled
consumer.  Cases differ in the weight format (GGUF Q8_0 / Q4_K / Q6_K, MLX
affine 4-bit), in the activation type (bf16, or f32 as candle runs GGUF
models), in the arithmetic (default, exact weights, candle's 8-bit
activations) and in the number of activation rows: 1 when decoding, a few when
verifying drafted tokens, tens for batches, hundreds to thousands for prompts.

Weights are made as GGUF block bytes (or MLX arrays) from N(0, 0.02) by the
plain min / max quantizers below, activations from N(0, 1).
"""
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "token-horizon_amd"))
import thq  # noqa: E402

FORMATS = {"q8_0": thq.Q8_0, "q4_k": thq.Q4_K, "q6_k": thq.Q6_K, "affine": thq.MLX_Q4}
MODES = {"default": thq.MODE_DEQUANT_F32, "exact": thq.MODE_EXACT_W, "q8act": thq.MODE_Q8ACT}
TYPES = {"bf16": torch.bfloat16, "f32": torch.float32}


def listed():
    return [
        # One small projection on f32 activations: a candle program's single
        # call, where launch and call cost count.
        {"name": "project_q8_0_f32_m1", "op": "matmul", "format": "q8_0", "m": 1, "n": 3072, "k": 1024, "x": "f32",
         "y": "f32", "mode": "default"},
        # One token through a decoder layer: the decode loop of a serving
        # program, which captures its step in a HIP graph.
        {"name": "decode_layer_q4_k_m1", "op": "layer", "format": "q4_k", "m": 1, "h": 4096, "i": 12288, "qkv": 6144,
         "x": "bf16", "y": "bf16", "mode": "default", "graph": True},
        # Verifying five drafted tokens + 1 in the engine's own format, with
        # the tile planes that its few-row kernels use.
        {"name": "verify_mlp_affine_m6", "op": "mlp", "format": "affine", "m": 6, "h": 5120, "i": 17408, "x": "bf16",
         "y": "bf16", "mode": "default", "tiles": True},
        # The same step of a candle program, on f32 activations.
        {"name": "verify_layer_q4_k_f32_m5", "op": "layer", "format": "q4_k", "m": 5, "h": 4096, "i": 12288,
         "qkv": 6144, "x": "f32", "y": "f32", "mode": "default"},
        # A prompt of no particular length.
        {"name": "prompt_layer_q4_k_m333", "op": "layer", "format": "q4_k", "m": 333, "h": 4096, "i": 12288,
         "qkv": 6144, "x": "bf16", "y": "bf16", "mode": "default"},
        # A chunk of a long prompt.
        {"name": "prompt_mlp_q4_k_m2048", "op": "mlp", "format": "q4_k", "m": 2048, "h": 4096, "i": 12288, "x": "bf16",
         "y": "bf16", "mode": "default"},
        # The down projection that a Q4_K_M file keeps in 6 bits.
        {"name": "prompt_down_q6_k_m512", "op": "matmul", "format": "q6_k", "m": 512, "n": 4096, "k": 12288,
         "x": "bf16", "y": "bf16", "mode": "default"},
        # A prompt in a candle program: f32 activations throughout.
        {"name": "prompt_mlp_q4_k_f32_m300", "op": "mlp", "format": "q4_k", "m": 300, "h": 4096, "i": 12288,
         "x": "f32", "y": "f32", "mode": "default"},
        # candle's default arithmetic (8-bit activations): one token, and a
        # prompt.
        {"name": "decode_layer_q4_k_q8act_m1", "op": "layer", "format": "q4_k", "m": 1, "h": 4096, "i": 12288,
         "qkv": 6144, "x": "f32", "y": "f32", "mode": "q8act"},
        {"name": "prompt_mlp_q4_k_q8act_m256", "op": "mlp", "format": "q4_k", "m": 256, "h": 4096, "i": 12288,
         "x": "f32", "y": "f32", "mode": "q8act"},
        # The LM head of a verify step over 8 sequences of 5 tokens, greedy.
        {"name": "head_q8_0_argmax_m40", "op": "head", "format": "q8_0", "m": 40, "n": 151936, "k": 4096, "x": "bf16",
         "mode": "default", "top": 0},
        # One sampled token off a 6-bit head.
        {"name": "head_q6_k_top32_m1", "op": "head", "format": "q6_k", "m": 1, "n": 151936, "k": 4096, "x": "bf16",
         "mode": "default", "top": 32},
    ]


def draw(rng):
    """One more case: rows from 1 to 2048, and weights from small projections to
    heads, ragged sizes among them.  None costs more than the listed case of
    its kind."""
    def spread(lo, hi):
        return int(round(lo * (hi / lo) ** rng.random()))

    op = rng.choice(["matmul", "matmul", "matmul", "mlp", "layer", "head"])
    if op == "head":
        fmt = rng.choice(["q8_0", "q6_k", "q4_k"])
        top = rng.choice([0, 0, 1, 20, 32, 64])
        return {"op": op, "format": fmt, "m": spread(1, 64 if fmt == "q4_k" else 40),
                "n": rng.choice([spread(32000, 151936), 32 * spread(1000, 4748)]), "k": 256 * rng.randint(4, 16),
                "x": "bf16", "mode": "default", "top": top}
    mode = rng.choice(["default", "default", "default", "exact", "q8act"])
    fmt = rng.choice(["q8_0", "q4_k"] if mode == "q8act" else ["q8_0", "q4_k", "q4_k", "q6_k", "affine"])
    x = rng.choice(["bf16", "bf16", "f32"])
    case = {"op": op, "format": fmt, "m": spread(1, 2048), "x": x, "y": x if x == "f32" else rng.choice(["bf16", "f32"]),
            "mode": mode}
    if op == "matmul":
        n = spread(512, 24576)
        case.update(n=rng.choice([n, (n + 127) // 128 * 128]), k=256 * spread(4, 68))
        size = case["n"] * case["k"]
    else:
        h = 256 * spread(4, 20)
        i = 256 * rng.randint(h // 256 * 2, h // 256 * 4)
        if op == "layer":
            case.update(qkv=h + 256 * rng.randint(1, h // 128))
        case.update(h=h, i=i)
        size = 3 * h * i + (case.get("qkv", -h) + h) * h
    # rows x weights of the largest listed case of the same arithmetic
    slow = 256 if mode == "q8act" else 300 if x == "f32" else 512 if mode == "exact" else 2048
    case["m"] = max(1, min(case["m"], slow * 3 * 12288 * 4096 // size))
    if fmt in ("q4_k", "affine") and 2 <= case["m"] <= 8 and rng.random() < 0.4:
        case["tiles"] = True
    return case


# ---------------------------------------------------------------------------- weights


def _rows(n, k):
    """Row ranges whose temporaries stay small."""
    step = max(1, (1 << 27) // k)
    return [(a, min(n, a + step)) for a in range(0, n, step)]


def _codes_q8_0(w):
    b = w.view(w.shape[0], -1, 32)
    d = (b.abs().amax(-1) / 127).half()
    q = torch.round(b / d.float().clamp_min(1e-12).unsqueeze(-1)).clamp(-127, 127)
    return d, q


def _codes_q4_k(w):
    b = w.view(w.shape[0], -1, 8, 32)
    low = b.amin(-1).clamp_max(0)
    s, m = (b.amax(-1) - low) / 15, -low
    d, dmin = (s.amax(-1, keepdim=True) / 63).half(), (m.amax(-1, keepdim=True) / 63).half()
    sc = torch.round(s / d.float()).clamp(1, 63)
    mm = torch.round(m / dmin.float()).clamp(0, 63)
    q = torch.round((b + (dmin.float() * mm).unsqueeze(-1)) / (d.float() * sc).unsqueeze(-1)).clamp(0, 15)
    return d, dmin, sc, mm, q


def _codes_q6_k(w):
    b = w.view(w.shape[0], -1, 16, 16)
    s = b.abs().amax(-1) / 31
    d = (s.amax(-1, keepdim=True) / 127).half()
    sc = torch.round(s / d.float()).clamp(1, 127)
    q = torch.round(b / (d.float() * sc).unsqueeze(-1)).clamp(-32, 31)
    return d, sc, q


def _codes_affine(w):
    b = w.view(w.shape[0], -1, 64)
    low = b.amin(-1)
    s, z = ((b.amax(-1) - low) / 15).bfloat16(), low.bfloat16()
    q = torch.round((b - z.float().unsqueeze(-1)) / s.float().unsqueeze(-1)).clamp(0, 15)
    return s, z, q


def _bytes(t):
    return t.contiguous().view(torch.uint8)


def _pack_q8_0(w):
    d, q = _codes_q8_0(w)
    return torch.cat([_bytes(d.unsqueeze(-1)), _bytes(q.to(torch.int8))], -1).view(-1)


def _pack_q4_k(w):
    d, dmin, sc, mm, q = _codes_q4_k(w)
    sc, mm, q = sc.to(torch.uint8), mm.to(torch.uint8), q.to(torch.uint8)
    q = q.view(*q.shape[:2], 4, 2, 32)
    head = [sc[..., :4] | ((sc[..., 4:] >> 4) << 6), mm[..., :4] | ((mm[..., 4:] >> 4) << 6),
            (sc[..., 4:] & 15) | ((mm[..., 4:] & 15) << 4)]
    nib = (q[..., 0, :] | (q[..., 1, :] << 4)).flatten(2)
    return torch.cat([_bytes(d), _bytes(dmin), *head, nib], -1).view(-1)


def _pack_q6_k(w):
    d, sc, q = _codes_q6_k(w)
    c = (q + 32).to(torch.uint8).view(q.shape[0], q.shape[1], 2, 4, 32)
    low, high = c & 15, c >> 4
    ql = torch.cat([low[..., 0, :] | (low[..., 2, :] << 4), low[..., 1, :] | (low[..., 3, :] << 4)], -1).flatten(2)
    qh = (high[..., 0, :] | (high[..., 1, :] << 2) | (high[..., 2, :] << 4) | (high[..., 3, :] << 6)).flatten(2)
    return torch.cat([ql, qh, _bytes(sc.to(torch.int8)), _bytes(d)], -1).view(-1)


def _pack_affine(w):
    s, z, q = _codes_affine(w)
    q = q.to(torch.uint8).view(w.shape[0], -1, 2)
    return _bytes(q[..., 0] | (q[..., 1] << 4)), _bytes(torch.cat([s, z], -1))


def _values(fmt, w):
    """What the codes stand for, in 64 bits."""
    if fmt == "q8_0":
        d, q = _codes_q8_0(w)
        v = d.double().unsqueeze(-1) * q.double()
    elif fmt == "q4_k":
        d, dmin, sc, mm, q = _codes_q4_k(w)
        v = (d.double() * sc.double()).unsqueeze(-1) * q.double() - (dmin.double() * mm.double()).unsqueeze(-1)
    elif fmt == "q6_k":
        d, sc, q = _codes_q6_k(w)
        v = (d.double() * sc.double()).unsqueeze(-1) * q.double()
    else:
        s, z, q = _codes_affine(w)
        v = s.double().unsqueeze(-1) * q.double() + z.double().unsqueeze(-1)
    return v.view(w.shape)


def _chunks(n, k, gen):
    for a, b in _rows(n, k):
        yield torch.randn((b - a, k), generator=gen, device="cuda") * 0.02


def _weight(fmt, n, k, gen):
    """A weight [n, k], loaded as a program loads a file's tensors."""
    if fmt == "affine":
        parts = [_pack_affine(w) for w in _chunks(n, k, gen)]
        return thq.QTensor.from_affine(torch.cat([p[0] for p in parts]), torch.cat([p[1] for p in parts]), n, k)
    pack = {"q8_0": _pack_q8_0, "q4_k": _pack_q4_k, "q6_k": _pack_q6_k}[fmt]
    return thq.QTensor.from_gguf_bytes(FORMATS[fmt], torch.cat([pack(w) for w in _chunks(n, k, gen)]), n, k)


def _shapes(case):
    """The weights of a case by name, in the order they are made: (rows, columns)."""
    if case["op"] in ("matmul", "head"):
        return {"w": (case["n"], case["k"])}
    h, i = case["h"], case["i"]
    mlp = {"gate_up": (2 * i, h), "down": (h, i)}
    return {"qkv": (case["qkv"], h), "o": (h, h), **mlp} if case["op"] == "layer" else mlp


def _inputs(case):
    """The activations of a case by name: the columns of each."""
    if case["op"] in ("matmul", "head"):
        return {"x": case["k"]}
    return {"x": case["h"], "attn": case["h"], "mlp": case["h"]} if case["op"] == "layer" else {"mlp": case["h"]}


def _activations(case, gen):
    return {name: torch.randn((case["m"], k), generator=gen, device="cuda").to(TYPES[case["x"]])
            for name, k in _inputs(case).items()}


# ---------------------------------------------------------------------------- passes


def prepare(case, seed):
    """A program's loaded weights, its activations and, where it captures its step, the graph."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    state = {"case": case, "w": {name: _weight(case["format"], n, k, gen) for name, (n, k) in _shapes(case).items()},
             **_activations(case, gen)}
    if case.get("tiles"):
        for w in state["w"].values():
            w.add_tiles()
    if case.get("graph"):
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _pass(state)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            state["out"] = _pass(state)
        state["graph"] = graph
    return state


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    return _pass(state)


def _pass(state):
    case, w = state["case"], state["w"]
    flags = MODES[case["mode"]]
    if case["op"] == "head":
        if case["top"]:
            logits, vals, idx = thq.matmul_topk(w["w"], state["x"], case["top"], want_logits=True, flags=flags)
            return {"logits": logits, "vals": vals, "idx": idx}
        logits, idx = thq.matmul_argmax(w["w"], state["x"], flags=flags)
        return {"logits": logits, "idx": idx}
    y = TYPES[case["y"]]
    if case["op"] == "matmul":
        return thq.matmul(w["w"], state["x"], y, flags)
    out = {}
    if case["mode"] == "q8act" and case["format"] == "q4_k" and case["op"] == "layer":
        # each input quantized once; the gate/up emits the down projection's operand
        out["qkv"] = thq.Q8Act(state["x"], thq.Q8_K).matmul(w["qkv"], y)
        out["o"] = thq.Q8Act(state["attn"], thq.Q8_K).matmul(w["o"], y)
        out["h"], operand = thq.Q8Act(state["mlp"], thq.Q8_K).gate_up_silu_emit(w["gate_up"], TYPES[case["x"]])
        out["down"] = operand.matmul(w["down"], y)
        return out
    if case["op"] == "layer":
        out["qkv"] = thq.matmul(w["qkv"], state["x"], y, flags)
        out["o"] = thq.matmul(w["o"], state["attn"], y, flags)
    out["h"] = thq.gate_up_silu(w["gate_up"], state["mlp"], TYPES[case["x"]], flags)
    out["down"] = thq.matmul(w["down"], out["h"], y, flags)
    return out


# ---------------------------------------------------------------------------- what it costs, and what it gives


def _outputs(case):
    """Bytes of the outputs of one pass."""
    m = case["m"]
    if case["op"] == "head":
        return 4 * m * case["n"] + (8 * m * case["top"] if case["top"] else 4 * m)
    size = 4 if case["y"] == "f32" else 2
    if case["op"] == "matmul":
        return size * m * case["n"]
    cols = case["h"] + (case["qkv"] + case["h"] if case["op"] == "layer" else 0)
    return size * m * cols + (4 if case["x"] == "f32" else 2) * m * case["i"]


def work(case):
    per = {"q8_0": 34 / 32, "q4_k": 144 / 256, "q6_k": 210 / 256, "affine": 144 / 256}[case["format"]]
    cells = sum(n * k for n, k in _shapes(case).values())
    x = case["m"] * sum(_inputs(case).values()) * (4 if case["x"] == "f32" else 2)
    return {"bytes": int(cells * per) + x + _outputs(case), "flops": 2 * case["m"] * cells}


def tolerance(case):
    """About four times what the paths show against exact().

    Exact weights with f32 sums are 1e-7 to 1.4e-6 off.  bf16 outputs add their
    own rounding, which two correct sums share but for a few values that lie
    between two neighbours (at most 2e-4 in all, one value in 2^8 at the most);
    the MLP rounds its gate and up sums so whatever the outputs' type, and with
    8-bit activations the down projection quantizes the result once more.
    Prompts on bf16 activations may round the weights to bf16: 2.3e-3 on a
    projection, 4.7e-3 behind the MLP."""
    exact_weights = case["mode"] != "default" or case["x"] == "f32" or case["op"] == "head" or case["m"] <= 16
    if not exact_weights:
        return {"rel": 0.02 if case["op"] != "matmul" else 0.01, "max": 0.2}
    if case["op"] == "head":
        return {"rel": 6e-6, "differ": 0.01}
    if case["op"] == "matmul" and case["y"] == "f32":
        return {"rel": 6e-6}
    return {"rel": 2e-3 if case["mode"] == "q8act" else 8e-4, "max": 0.03}


def _silu_mul(gu, to):
    """silu(bf16(g)) * bf16(u) of [gate | up] columns, as the type of activations that the down projection reads."""
    g, u = gu.float().bfloat16().double().chunk(2, -1)
    return (g * torch.sigmoid(g) * u).float().to(to).double()


def _as_q8_0(x):
    """candle's 8-bit activations of a Q8_0 weight, as 64-bit values."""
    b = x.float().view(x.shape[0], -1, 32)
    d = b.abs().amax(-1, keepdim=True) / 127
    v = b * torch.where(d != 0, 1 / d, torch.zeros_like(d))
    q = torch.sign(v) * torch.floor(v.abs().double() + 0.5).float()
    return (q.double() * d.half().double()).view(x.shape)


def _as_q8_k(x):
    """candle's 8-bit activations of a Q4_K weight, as 64-bit values."""
    b = x.float().view(x.shape[0], -1, 256)
    top = torch.gather(b, -1, b.abs().argmax(-1, keepdim=True))
    scale = torch.where(top != 0, -128 / top, torch.zeros_like(top))
    v = scale * b
    q = (torch.sign(v) * torch.floor(v.abs().double() + 0.5).float()).clamp_max(127)
    d = torch.where(top != 0, 1 / scale, torch.zeros_like(scale))
    return (q.double() * d.double()).view(x.shape)


def exact(case, seed):
    """run()'s outputs in 64 bits (the head's indices have no such value)."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    fmt = case["format"]
    w = {name: torch.cat([_values(fmt, c) for c in _chunks(n, k, gen)]) for name, (n, k) in _shapes(case).items()}
    x = _activations(case, gen)

    def project(name, v):
        v = v.double()
        if case["mode"] == "q8act":
            v = _as_q8_0(v) if fmt == "q8_0" else _as_q8_k(v)
        return v @ w[name].T

    if case["op"] == "head":
        logits = project("w", x["x"])
        return {"logits": logits, "vals": logits.topk(case["top"]).values, "idx": None} if case["top"] else \
            {"logits": logits, "idx": None}
    if case["op"] == "matmul":
        return project("w", x["x"])
    out = {"qkv": project("qkv", x["x"]), "o": project("o", x["attn"])} if case["op"] == "layer" else {}
    out["h"] = _silu_mul(project("gate_up", x["mlp"]), TYPES[case["x"]])
    out["down"] = project("down", out["h"])
    return out
