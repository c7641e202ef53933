"""The work a program has this framework do, as cases to time and to compare.

Each case is one pass through the public entry points of ``lightbulb_amd.quantized``
over weights in their GGUF block layout.  The shapes are the Llama-3-8B projections the
benchmark uses, the same kinds of call at other widths and generic odd sizes:

* ``linear``   one projection (``QMatMul.forward``): decode, short prompts, prefill,
               weights whose k is no multiple of 256, and dense F16 / BF16 / F32 weights
* ``head``     the final RMS norm and the LM head
* ``layer``    the projections of one layer through the fused call sites
* ``mlp``      the gate / up / SiLU product and the down projection of a prefill chunk
* ``embed``    the token embedding of a prompt from the quantised table
* ``convert``  a weight file's tensor turned from one type into another

Weights are blocks of random codes and scales (the codes bell-shaped and the values of
mean zero, as quantised weights are); activations are normal with 1 % of the entries
20 times as large, as a transformer's are.
"""
from __future__ import annotations

import math

import torch

from lightbulb_amd import quantized as qz

T = qz.GgmlDType
DENSE = ("F32", "F16", "BF16")
EPS = 1e-5


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------
def listed() -> list[dict]:
    return [
        # the smallest projection of a token step: latency and launches count
        {"name": "k_proj_decode", "op": "linear", "type": "Q4K", "n": 1024, "k": 4096, "m": 1},
        # one layer of the Q4_K_M mix for one token of one sequence
        {"name": "layer_decode", "op": "layer", "mix": "Q4_K_M", "hidden": 4096, "kv": 1024, "inter": 14336, "m": 1},
        # the LM head of the same token: the longest single weight stream
        {"name": "head_decode", "op": "head", "type": "Q6K", "n": 128256, "k": 4096, "m": 1},
        # the layer with 32 sequences batched
        {"name": "layer_batch32", "op": "layer", "mix": "Q4_K_M", "hidden": 4096, "kv": 1024, "inter": 14336, "m": 32},
        # a short prompt of no round length through a wide-k projection
        {"name": "down_prompt100", "op": "linear", "type": "Q5K", "n": 4096, "k": 14336, "m": 100},
        # a prefill chunk through the MLP
        {"name": "mlp_prefill512", "op": "mlp", "type": "Q4K", "hidden": 4096, "inter": 14336, "m": 512},
        # a long prompt, or several together, through the MLP
        {"name": "mlp_prefill4096", "op": "mlp", "type": "Q4K", "hidden": 4096, "inter": 14336, "m": 4096},
        # a prompt of no round length through the attention projection of a Q8_0 file
        {"name": "q8_prompt333", "op": "linear", "type": "Q8_0", "n": 4096, "k": 4096, "m": 333},
        # a width that is no multiple of 256: such files hold 32-value blocks throughout
        {"name": "odd_width_prompt200", "op": "linear", "type": "Q8_0", "n": 5760, "k": 2880, "m": 200},
        # a file with unquantised weights: candle's f32 matmul
        {"name": "dense_f16_prefill512", "op": "linear", "type": "F16", "n": 4096, "k": 4096, "m": 512},
        # requantising a file's tensor: blocks -> f32 -> blocks
        {"name": "convert_q8_0_q4k", "op": "convert", "type": "Q8_0", "to": "Q4K", "n": 4096, "k": 4096},
        # the embedding of a prompt
        {"name": "embed_prompt2048", "op": "embed", "type": "Q4K", "n": 128256, "k": 4096, "count": 2048},
    ]


def _log_int(rng, lo: int, hi: int, step: int = 1) -> int:
    """A whole number of `step`s in [lo, hi], spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi + step)))
    return max(lo, min(hi, int(v) // step * step))


def _rows(rng) -> int:
    """Rows of x: one token, a batch of sequences, a prompt, a prefill chunk."""
    return 1 if rng.random() < 0.2 else _log_int(rng, 2, 2048)


def draw(rng) -> dict:
    op = rng.choice(("linear", "linear", "odd", "dense", "head", "layer", "mlp", "embed", "convert"))
    if op == "linear":
        return {"op": "linear", "type": rng.choice(("Q4K", "Q5K", "Q6K", "Q8_0", "Q4_0", "Q5_0")),
                "n": _log_int(rng, 512, 16384), "k": _log_int(rng, 1024, 14336, 256), "m": _rows(rng)}
    if op == "odd":
        k = _log_int(rng, 1024, 8192, 32)
        return {"op": "linear", "type": rng.choice(("Q8_0", "Q4_0", "Q5_0")), "n": _log_int(rng, 512, 8192),
                "k": k + 32 if k % 256 == 0 else k, "m": _rows(rng)}
    if op == "dense":
        return {"op": "linear", "type": rng.choice(DENSE), "n": _log_int(rng, 512, 8192),
                "k": _log_int(rng, 512, 8192, 8), "m": _rows(rng)}
    if op == "head":
        return {"op": "head", "type": rng.choice(("Q6K", "Q8_0", "Q4K")), "n": _log_int(rng, 32000, 128256),
                "k": _log_int(rng, 2048, 4096, 256), "m": _log_int(rng, 1, 8)}
    if op == "layer":
        hidden = _log_int(rng, 1024, 8192, 256)
        return {"op": "layer", "mix": rng.choice(("Q4_K_M", "Q5_K_M", "Q6_K", "Q8_0")), "hidden": hidden,
                "kv": _log_int(rng, 256, 1024, 64), "inter": _log_int(rng, 2 * hidden, 16384, 256),
                "m": _log_int(rng, 1, 64)}
    if op == "mlp":
        hidden = _log_int(rng, 1024, 4096, 256)
        return {"op": "mlp", "type": rng.choice(("Q4K", "Q5K", "Q6K", "Q8_0")), "hidden": hidden,
                "inter": _log_int(rng, 2 * hidden, 14336, 256), "m": _log_int(rng, 128, 4096)}
    if op == "embed":
        return {"op": "embed", "type": rng.choice(("Q4K", "Q6K", "Q8_0", "F16")), "n": _log_int(rng, 32000, 128256),
                "k": _log_int(rng, 1024, 4096, 256), "count": _log_int(rng, 1, 4096)}
    return {"op": "convert", "type": rng.choice(("Q8_0", "F16", "BF16")), "to": rng.choice(("Q4K", "Q5K", "Q6K", "Q8_0")),
            "n": _log_int(rng, 512, 8192), "k": _log_int(rng, 1024, 8192, 256)}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _codes(g, nb: int, per: int, top: int) -> torch.Tensor:
    """Bell-shaped unsigned codes 0..top, [nb, per] uint8."""
    c = torch.randn(nb, per, generator=g, device="cuda")
    return c.mul_((top + 1) / 5.0).add_(top / 2.0).round_().clamp_(0, top).to(torch.uint8)


def _f16_bytes(v: torch.Tensor) -> torch.Tensor:
    return v.to(torch.float16).reshape(-1, 1).view(torch.uint8)


def _scale(g, nb: int, typical: float) -> torch.Tensor:
    return typical * (0.7 + 0.6 * torch.rand(nb, generator=g, device="cuda"))


def _six_bit(sc: torch.Tensor, mn: torch.Tensor) -> torch.Tensor:
    """The 12 bytes of eight 6-bit scales and mins."""
    lo = (sc[:, :4] & 63) | ((sc[:, 4:] >> 4) << 6)
    hi = (mn[:, :4] & 63) | ((mn[:, 4:] >> 4) << 6)
    return torch.cat([lo, hi, (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)], 1)


def _blocks(g, name: str, n: int, k: int) -> torch.Tensor:
    """n x k weights of the type, as flat block bytes; values of about 0.02."""
    if name in DENSE:
        w = torch.randn(n * k, generator=g, device="cuda").mul_(0.02)
        return w.to({"F32": torch.float32, "F16": torch.float16, "BF16": torch.bfloat16}[name]).view(torch.uint8)
    nb = n * (k // T[name].block_size())
    if name in ("Q4K", "Q5K"):
        top = 15 if name == "Q4K" else 31
        q = _codes(g, nb, 256, top)
        sc = torch.randint(24, 64, (nb, 8), generator=g, device="cuda", dtype=torch.uint8)
        mn = (sc.to(torch.int16) + torch.randint(-3, 4, (nb, 8), generator=g, device="cuda")).clamp_(0, 63).to(torch.uint8)
        d = _scale(g, nb, 0.02 / (42 * (top + 1) / 5.0))
        p = q.view(nb, 4, 2, 32)
        qs = ((p[:, :, 0] & 15) | ((p[:, :, 1] & 15) << 4)).reshape(nb, 128)
        parts = [_f16_bytes(d), _f16_bytes(d * (top / 2.0)), _six_bit(sc, mn)]
        if name == "Q5K":
            qh = torch.zeros(nb, 32, dtype=torch.uint8, device="cuda")
            for c in range(4):
                qh |= ((p[:, c, 0] >> 4) << (2 * c)) | ((p[:, c, 1] >> 4) << (2 * c + 1))
            parts.append(qh)
        return torch.cat([*parts, qs], 1).reshape(-1)
    if name == "Q6K":
        q = _codes(g, nb, 256, 63).view(nb, 2, 4, 32)
        ql = torch.stack([(q[:, :, 0] & 15) | ((q[:, :, 2] & 15) << 4), (q[:, :, 1] & 15) | ((q[:, :, 3] & 15) << 4)], 2)
        qh = (q[:, :, 0] >> 4) | ((q[:, :, 1] >> 4) << 2) | ((q[:, :, 2] >> 4) << 4) | ((q[:, :, 3] >> 4) << 6)
        sc = torch.randint(40, 128, (nb, 16), generator=g, device="cuda", dtype=torch.int8)
        sc = torch.where(torch.rand(nb, 16, generator=g, device="cuda") < 0.5, -sc, sc)
        d = _scale(g, nb, 0.02 / (80 * 64 / 5.0))
        return torch.cat([ql.reshape(nb, 128), qh.reshape(nb, 64), sc.view(torch.uint8), _f16_bytes(d)], 1).reshape(-1)
    if name == "Q8_0":
        q = _codes(g, nb, 32, 254).to(torch.int16).sub_(127).to(torch.int8).view(torch.uint8)
        return torch.cat([_f16_bytes(_scale(g, nb, 0.02 / 51)), q], 1).reshape(-1)
    top = 15 if name == "Q4_0" else 31
    q = _codes(g, nb, 32, top)
    parts = [_f16_bytes(_scale(g, nb, 0.02 / ((top + 1) / 5.0)))]
    if name == "Q5_0":
        bit = (q >> 4).view(nb, 4, 8) << torch.arange(8, dtype=torch.uint8, device="cuda")
        parts.append(bit.sum(2, dtype=torch.uint8))
    parts.append((q[:, :16] & 15) | ((q[:, 16:] & 15) << 4))
    return torch.cat(parts, 1).reshape(-1)


def _tensor(g, name: str, n: int, k: int) -> "qz.QTensor":
    return qz.QTensor(_blocks(g, name, n, k), T[name], (n, k))


def _matmul(g, name: str, n: int, k: int) -> "qz.QMatMul":
    return qz.QMatMul.from_qtensor(_tensor(g, name, n, k))


def _x(g, m: int, k: int) -> torch.Tensor:
    """Activations [1, m, k], as a program holds them (batch, sequence, width)."""
    x = torch.randn(1, m, k, generator=g, device="cuda")
    return torch.where(torch.rand(1, m, k, generator=g, device="cuda") < 0.01, x * 20.0, x)


def _norm(g, k: int) -> torch.Tensor:
    return 1.0 + 0.1 * torch.randn(k, generator=g, device="cuda")


def _layer_types(mix: str) -> dict[str, str]:
    """The types of a file's mix: the _M mixes keep v and (here) down in Q6_K."""
    base = {"Q4_K_M": "Q4K", "Q5_K_M": "Q5K", "Q6_K": "Q6K", "Q8_0": "Q8_0"}[mix]
    up = "Q6K" if mix.endswith("_M") else base
    return {"q": base, "k": base, "v": up, "o": base, "gate": base, "up": base, "down": up}


def _layer_shapes(c: dict) -> dict[str, tuple[int, int]]:
    h, kv, inter = c["hidden"], c["kv"], c["inter"]
    return {"q": (h, h), "k": (kv, h), "v": (kv, h), "o": (h, h), "gate": (inter, h), "up": (inter, h), "down": (h, inter)}


def prepare(case: dict, seed: int) -> dict:
    g, op = _gen(seed), case["op"]
    s = {"op": op}
    if op == "linear":
        s["w"] = qz.QuantizableLinear.from_qmatmul(_matmul(g, case["type"], case["n"], case["k"]))
        s["x"] = _x(g, case["m"], case["k"])
    elif op == "head":
        s["w"], s["x"] = _matmul(g, case["type"], case["n"], case["k"]), _x(g, case["m"], case["k"])
        s["norm"] = _norm(g, case["k"])
    elif op == "layer":
        types = _layer_types(case["mix"])
        s["w"] = {p: _matmul(g, types[p], n, k) for p, (n, k) in _layer_shapes(case).items()}
        s["same"] = types["v"] == types["q"]
        s["x"], s["attn"], s["mid"] = (_x(g, case["m"], case["hidden"]) for _ in range(3))
        s["norm1"], s["norm2"] = _norm(g, case["hidden"]), _norm(g, case["hidden"])
    elif op == "mlp":
        h, inter = case["hidden"], case["inter"]
        s["gate"], s["up"] = _matmul(g, case["type"], inter, h), _matmul(g, case["type"], inter, h)
        s["down"], s["x"], s["norm"] = _matmul(g, case["type"], h, inter), _x(g, case["m"], h), _norm(g, h)
    elif op == "embed":
        s["w"] = qz.QEmbedding(_tensor(g, case["type"], case["n"], case["k"]))
        s["ids"] = torch.randint(0, case["n"], (1, case["count"]), generator=g, device="cuda")
    else:
        s["w"], s["to"] = _tensor(g, case["type"], case["n"], case["k"]), T[case["to"]]
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(s: dict):
    op = s["op"]
    if op == "linear":
        return s["w"].forward(s["x"])
    if op == "head":
        return qz.rmsnorm_qmatmul_group([s["w"]], s["x"], s["norm"], EPS)[0]
    if op == "layer":
        w = s["w"]
        if s["same"]:
            q, k, v = qz.rmsnorm_qmatmul_group([w["q"], w["k"], w["v"]], s["x"], s["norm1"], EPS)
        else:
            q, k = qz.rmsnorm_qmatmul_group([w["q"], w["k"]], s["x"], s["norm1"], EPS)
            v, = qz.rmsnorm_qmatmul_group([w["v"]], s["x"], s["norm1"], EPS)
        o = w["o"].forward(s["attn"])
        h = qz.rmsnorm_gate_up_silu(w["gate"], w["up"], s["mid"], s["norm2"], EPS)
        return {"q": q, "k": k, "v": v, "o": o, "h": h, "down": w["down"].forward(h)}
    if op == "mlp":
        h = qz.rmsnorm_gate_up_silu(s["gate"], s["up"], s["x"], s["norm"], EPS)
        return {"h": h, "down": s["down"].forward(h)}
    if op == "embed":
        return s["w"].forward(s["ids"])
    f = s["w"].dequantize()
    return {"f32": f, "blocks": qz.QTensor.quantize(f, s["to"]).data}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _bytes(name: str, n: int, k: int) -> int:
    return n * (k // T[name].block_size()) * T[name].block_bytes()


def work(case: dict) -> dict:
    op = case["op"]
    if op in ("linear", "head"):
        n, k, m = case["n"], case["k"], case["m"]
        return {"bytes": _bytes(case["type"], n, k) + 4 * m * (n + k), "flops": 2 * m * n * k}
    if op == "layer":
        types, m = _layer_types(case["mix"]), case["m"]
        shapes = _layer_shapes(case)
        io = 3 * case["hidden"] + sum(n for n, _ in shapes.values()) - shapes["up"][0] + 2 * case["hidden"]
        return {"bytes": sum(_bytes(types[p], n, k) for p, (n, k) in shapes.items()) + 4 * m * io,
                "flops": 2 * m * sum(n * k for n, k in shapes.values())}
    if op == "mlp":
        h, inter, m = case["hidden"], case["inter"], case["m"]
        return {"bytes": 3 * _bytes(case["type"], h, inter) + 4 * m * (2 * h + inter), "flops": 6 * m * h * inter}
    if op == "embed":
        return {"bytes": _bytes(case["type"], case["count"], case["k"]) + 8 * case["count"] + 4 * case["count"] * case["k"],
                "flops": 0}
    n, k = case["n"], case["k"]
    return {"bytes": _bytes(case["type"], n, k) + 4 * n * k + _bytes(case["to"], n, k), "flops": 0}


def tolerance(case: dict):
    op = case["op"]
    if op in ("embed", "convert"):
        return "exact"
    if op == "linear" and case["type"] in DENSE:
        return {"rel": 1e-5, "max": 1e-3}  # f32 sums in another order
    if op in ("layer", "mlp"):
        # the product h is quantised to 8 bits for down: a last-bit change of h moves codes to
        # their neighbour, whose step is 1/127 of the block's largest value
        return {"rel": 1e-2, "max": 0.4}
    if op == "head":
        return {"rel": 1e-3, "max": 4e-2}  # codes of the normalised x that lie at a tie
    # 8-bit codes times dequantised weights: integer sums (m <= 8) or fp16 operands
    return {"rel": 1.6e-3, "max": 6e-2}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _f16(b: torch.Tensor) -> torch.Tensor:
    return b.contiguous().view(torch.float16).to(torch.float64)


def _dequantized(name: str, raw: torch.Tensor, n: int, k: int) -> torch.Tensor:
    """f64 [n, k] from block bytes."""
    if name in DENSE:
        return raw.view({"F32": torch.float32, "F16": torch.float16, "BF16": torch.bfloat16}[name]).to(torch.float64).view(n, k)
    b = raw.view(-1, T[name].block_bytes())
    nb = b.shape[0]
    if name in ("Q4K", "Q5K"):
        s = b[:, 4:16]
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1).to(torch.float64)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).to(torch.float64)
        qs = b[:, -128:].reshape(nb, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2)
        if name == "Q5K":
            shift = torch.arange(8, dtype=torch.uint8, device=b.device).view(1, 4, 2, 1)
            q = q | (((b[:, 16:48].reshape(nb, 1, 1, 32) >> shift) & 1) << 4)
        q = q.reshape(nb, 8, 32).to(torch.float64)
        w = (_f16(b[:, 0:2]) * sc).unsqueeze(2) * q - (_f16(b[:, 2:4]) * mn).unsqueeze(2)
    elif name == "Q6K":
        ql, qh = b[:, :128].reshape(nb, 2, 2, 32), b[:, 128:192].reshape(nb, 2, 32)
        quarters = [((ql[:, :, s & 1] >> (4 * (s >> 1))) & 15) | (((qh >> (2 * s)) & 3) << 4) for s in range(4)]
        q = torch.stack(quarters, 2).reshape(nb, 16, 16).to(torch.float64) - 32.0
        w = (_f16(b[:, 208:210]) * b[:, 192:208].contiguous().view(torch.int8).to(torch.float64)).unsqueeze(2) * q
    elif name == "Q8_0":
        w = _f16(b[:, :2]) * b[:, 2:].contiguous().view(torch.int8).to(torch.float64)
    else:
        q = torch.cat([b[:, -16:] & 15, b[:, -16:] >> 4], 1)
        if name == "Q5_0":
            bit = (b[:, 2:6].unsqueeze(2) >> torch.arange(8, dtype=torch.uint8, device=b.device)) & 1
            q = q | (bit.reshape(nb, 32) << 4)
        w = _f16(b[:, :2]) * (q.to(torch.float64) - (8.0 if name == "Q4_0" else 16.0))
    return w.reshape(n, k)


def _round(v: torch.Tensor) -> torch.Tensor:
    return torch.trunc(v + torch.copysign(torch.full_like(v, 0.5), v))


def _quantized(name: str, x: torch.Tensor) -> torch.Tensor:
    """x [m, k] as the projection sees it, in f64: its 8-bit codes (formed in f32) times their scale."""
    x = x.to(torch.float32)
    if name in DENSE:
        return x.to(torch.float64)
    if name in ("Q4K", "Q5K", "Q6K"):
        v = x.reshape(x.shape[0], -1, 256)
        big = v.gather(2, v.abs().argmax(2, keepdim=True))
        inv = torch.where(big == 0, torch.zeros_like(big), -128.0 / big)
        d = torch.where(big == 0, torch.zeros_like(big), 1.0 / inv)
        q = _round(v * inv).clamp(max=127.0)
    else:
        v = x.reshape(x.shape[0], -1, 32)
        d = v.abs().amax(2, keepdim=True) / 127.0
        q = _round(v * torch.where(d == 0, torch.zeros_like(d), 1.0 / d)).clamp(-128.0, 127.0)
        d = d.to(torch.float16)
    return (q.to(torch.float64) * d.to(torch.float64)).reshape(x.shape)


def _forward(w: "qz.QMatMul", x: torch.Tensor) -> torch.Tensor:
    t = w.qtensor()
    (n, k), name = t.shape(), T(t.dtype()).name
    a, parts = _quantized(name, x.reshape(-1, k)), []
    per = t.data.numel() // n
    for r in range(0, n, 16384):  # a part of the weight's rows at a time
        e = min(n, r + 16384)
        parts.append(a @ _dequantized(name, t.data[r * per:e * per], e - r, k).t().contiguous())
    return torch.cat(parts, 1).reshape(*x.shape[:-1], n)


def _rms(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    x = x.to(torch.float64)
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.to(torch.float64)


def _gate_up(gate, up, x: torch.Tensor) -> torch.Tensor:
    g = _forward(gate, x)
    return g / (1.0 + torch.exp(-g)) * _forward(up, x)


def exact(case: dict, seed: int):
    s, op = prepare(case, seed), case["op"]
    if op == "linear":
        return _forward(s["w"].inner, s["x"])
    if op == "head":
        return _forward(s["w"], _rms(s["x"], s["norm"]))
    if op == "layer":
        w, xn = s["w"], _rms(s["x"], s["norm1"])
        h = _gate_up(w["gate"], w["up"], _rms(s["mid"], s["norm2"]))
        return {**{p: _forward(w[p], xn) for p in "qkv"}, "o": _forward(w["o"], s["attn"]), "h": h,
                "down": _forward(w["down"], h)}
    if op == "mlp":
        h = _gate_up(s["gate"], s["up"], _rms(s["x"], s["norm"]))
        return {"h": h, "down": _forward(s["down"], h)}
    if op == "embed":
        t = s["w"]._qmatmul.qtensor()
        (n, k), ids = t.shape(), s["ids"].reshape(-1)
        rows = t.data.view(n, -1)[ids].reshape(-1)
        return _dequantized(case["type"], rows, ids.numel(), k).reshape(*s["ids"].shape, k)
    return {"f32": _dequantized(case["type"], s["w"].data, case["n"], case["k"]), "blocks": None}
