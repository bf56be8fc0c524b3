"""The work that programs on this library have it do, as cases to time and compare.

A case is a dict of plain values; `op` names the call it makes:

  gemv    one decode mat-vec of S <= 8 tokens (tc_gemv)
  layer   a decode step of one token through several transformer layers, four
          launches each (q/k/v, o, gate/up with SwiGLU, down), issued as one
          graph replay, as a serving loop issues it
  mixed   one token through a mixed-quant block: IQ3_XXS gate/up, Q6_K down
          and the Q6_K LM head (returns the logits)
  gemm    one prefill product of M tokens (tc_gemm)
  moe     a mixture-of-experts block: router, then expert FFN (Q4_K experts)
  encode  fp32 weights to GGUF blocks (tc_encode)

Weights are raw GGUF blocks with random quants and scales of a size that
gives weights of standard deviation about 0.02; activations are N(0,1) fp32.
Matrices are [out][in].
"""
import math
import os
import re
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "tinycoder-inference_amd"))
import tc_hip  # noqa: E402

DEV = "cuda:0"
GRID_DIR = os.path.join(os.getcwd(), "tinycoder-inference_amd", "csrc")

# Types whose products take fp32 activations as they are; the others quantize
# them (Q8_0 weights: 32-wide blocks, the rest: 256-wide) as the entry points say.
FP32_X = ("IQ2_XS", "IQ4_NL", "Q5_0")
ENCODED = ("Q4_K", "Q5_K", "Q6_K", "Q8_0")

# Where a block holds its fp16 scale(s), and the size that makes the weights
# come out at about 0.02.
SCALES = {
    "Q8_0": [(0, 2.7e-4)],
    "Q2_K": [(80, 1.6e-3), (82, 2.4e-3)],
    "Q3_K": [(108, 4.8e-4)],
    "Q4_K": [(0, 1.2e-4), (2, 9.0e-4)],
    "Q5_K": [(0, 6.0e-5), (2, 9.3e-4)],
    "Q6_K": [(208, 2.0e-5)],
    "IQ2_XS": [(0, 5.0e-4)],
    "IQ3_XXS": [(0, 2.0e-4)],
    "IQ3_S": [(0, 1.6e-4)],
    "IQ2_S": [(0, 5.0e-4)],
    "IQ4_XS": [(0, 1.6e-5)],
    "IQ4_NL": [(0, 2.9e-4)],
    "Q5_0": [(0, 2.2e-3)],
}


def listed():
    return [
        # The smallest call: one 4096-wide projection of a small Q8_0 model, one token, called eagerly.
        {"name": "gemv_q8_0_4096", "op": "gemv", "type": "Q8_0", "S": 1, "rows": 4096, "cols": 4096},
        # The decode step of a 7B model: four of its layers, one token.
        {"name": "layer_q4_k_7b", "op": "layer", "type": "Q4_K", "layers": 4, "hidden": 3584, "kv": 512, "ff": 18944},
        # The same model in a mixed-quant file: FFN of a layer and the 152064-word LM head.
        {"name": "mixed_q6_k_iq3_xxs_7b", "op": "mixed", "hidden": 3584, "ff": 18944, "vocab": 152064},
        # Several sequences decoded together, an odd number of them: the FFN up projection for 5 tokens.
        {"name": "gemv_q5_k_5tok", "op": "gemv", "type": "Q5_K", "S": 5, "rows": 18944, "cols": 3584},
        # A short prompt (or one chunk of a long one) through an FFN projection.
        {"name": "gemm_q4_k_m128", "op": "gemm", "type": "Q4_K", "M": 128, "rows": 17408, "cols": 5120},
        # A long prompt through the FFN down projection.
        {"name": "gemm_q4_k_m2048", "op": "gemm", "type": "Q4_K", "M": 2048, "rows": 5120, "cols": 17408},
        # Q8_0 of a width that is no multiple of 256, with odd rows and tokens.
        {"name": "gemm_q8_0_ragged", "op": "gemm", "type": "Q8_0", "M": 333, "rows": 4001, "cols": 2880},
        # A low-bit file's prompt: most matrices of a 3-bit K-quant file are Q3_K.
        {"name": "gemm_q3_k_m512", "op": "gemm", "type": "Q3_K", "M": 512, "rows": 18944, "cols": 3584},
        # A type whose products take the activations unquantized, a short ragged prompt, the wide down projection.
        {"name": "gemm_iq4_nl_m100", "op": "gemm", "type": "IQ4_NL", "M": 100, "rows": 3584, "cols": 18944},
        # One token through a 128-expert block, as a decode step has it.
        {"name": "moe_1tok", "op": "moe", "T": 1, "E": 128, "K": 8, "hidden": 2048, "ff": 768},
        # A prompt through the same block.
        {"name": "moe_1024tok", "op": "moe", "T": 1024, "E": 128, "K": 8, "hidden": 2048, "ff": 768},
        # One FFN matrix of a model quantized on load.
        {"name": "encode_q4_k", "op": "encode", "type": "Q4_K", "rows": 18944, "cols": 3584},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _wide(rng, lo, hi):
    return max(1, int(round(_log(rng, lo, hi) / 256))) * 256


def draw(rng):
    op = rng.choice(["gemv", "gemv", "layer", "mixed", "gemm", "gemm", "gemm", "moe", "moe", "encode"])
    types = sorted(SCALES)
    if op in ("gemv", "gemm"):
        t = rng.choice(types)
        cols = _wide(rng, 512, 18944)
        if t == "Q8_0" and rng.random() < 0.5:
            cols = max(16, _log(rng, 16, 592)) * 32
        if op == "gemv":
            rows = min(_log(rng, 256, 152064), 545_000_000 // cols)
            return {"op": op, "type": t, "S": rng.randint(1, 8), "rows": rows, "cols": cols}
        rows = _log(rng, 256, 18944)
        M = max(9, min(_log(rng, 9, 2048), 2048 * 5120 * 17408 // (rows * cols)))
        return {"op": op, "type": t, "M": M, "rows": rows, "cols": cols}
    if op == "layer":
        return {"op": op, "type": rng.choice(["Q4_K", "Q4_K", "Q5_K", "Q6_K", "Q8_0", "Q3_K", "IQ4_XS"]), "layers": rng.randint(1, 4),
                "hidden": _wide(rng, 1024, 5120), "kv": 128 * rng.randint(1, 8), "ff": _wide(rng, 2048, 18944)}
    if op == "mixed":
        return {"op": op, "hidden": _wide(rng, 1024, 5120), "ff": _wide(rng, 2048, 18944), "vocab": _log(rng, 16000, 106000)}
    if op == "moe":
        E = rng.choice([8, 16, 60, 64, 128, 128, 256])
        K = rng.randint(1, 8)
        hidden, ff = _wide(rng, 1024, 4096), _wide(rng, 512, 2048)
        while E * hidden * ff > 128 * 2048 * 2048:
            E //= 2
        K = min(K, E)
        return {"op": op, "T": _log(rng, 1, 2048), "E": E, "K": K, "hidden": hidden, "ff": ff}
    return {"op": op, "type": rng.choice(ENCODED), "rows": _log(rng, 256, 18944), "cols": _wide(rng, 512, 3584)}


# ---- inputs ----------------------------------------------------------------------


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 1_000_003 + 17)
    return g


def _blocks(t, g, rows, cols):
    q = getattr(tc_hip, t)
    n = rows * cols // tc_hip.BLOCK_SIZE[q]
    b = torch.randint(0, 256, (n, tc_hip.TYPE_SIZE[q]), dtype=torch.uint8, device=DEV, generator=g)
    if t == "Q8_0":  # its encoders write -127..127
        b[:, 2:] = torch.where(b[:, 2:] == 128, 129, b[:, 2:])
    for off, size in SCALES[t]:
        d = (torch.rand(n, device=DEV, generator=g) + 0.5) * size
        b[:, off:off + 2] = d.to(torch.float16).view(torch.uint8).view(n, 2)
    return b.view(-1)


def _randn(g, *shape):
    return torch.randn(*shape, device=DEV, dtype=torch.float32, generator=g)


_LIB = None


def _lib():
    global _LIB
    if _LIB is None:
        _LIB = tc_hip.Library()
    return _LIB


def _layer_shapes(case):
    h, kv, ff = case["hidden"], case["kv"], case["ff"]
    return {"q": (h, h), "k": (kv, h), "v": (kv, h), "o": (h, h), "gate": (ff, h), "up": (ff, h), "down": (h, ff)}


def _inputs(case, seed):
    """Weights and activations of a case, in a dict."""
    g, op = _gen(seed), case["op"]
    if op in ("gemv", "gemm"):
        n = case["S"] if op == "gemv" else case["M"]
        return {"w": _blocks(case["type"], g, case["rows"], case["cols"]), "x": _randn(g, n, case["cols"])}
    if op == "layer":
        layers = []
        for _ in range(case["layers"]):
            one = {k: _blocks(case["type"], g, r, c) for k, (r, c) in _layer_shapes(case).items()}
            one.update(x=_randn(g, 1, case["hidden"]), attn=_randn(g, 1, case["hidden"]),
                       x2=_randn(g, 1, case["hidden"]), h=_randn(g, 1, case["ff"]))
            layers.append(one)
        return {"layers": layers}
    if op == "mixed":
        h, ff = case["hidden"], case["ff"]
        return {"gate": _blocks("IQ3_XXS", g, ff, h), "up": _blocks("IQ3_XXS", g, ff, h), "down": _blocks("Q6_K", g, h, ff),
                "head": _blocks("Q6_K", g, case["vocab"], h), "x": _randn(g, 1, h), "h": _randn(g, 1, ff), "last": _randn(g, 1, h)}
    if op == "moe":
        E, H, F = case["E"], case["hidden"], case["ff"]
        return {"gate": _blocks("Q4_K", g, E * F, H), "up": _blocks("Q4_K", g, E * F, H), "down": _blocks("Q4_K", g, E * H, F),
                "router": _randn(g, E, H) / math.sqrt(H), "x": _randn(g, case["T"], H)}
    # weights whose rows differ in size, as a model's do
    std = 0.02 * torch.exp(torch.rand(case["rows"], 1, device=DEV, generator=g) * 1.6)
    return {"x": _randn(g, case["rows"], case["cols"]) * std}


def prepare(case, seed):
    state = {"case": case, "lib": _lib(), "in": _inputs(case, seed)}
    if case["op"] == "layer":
        # The step is captured once and replayed, as a serving loop does.
        rows = {k: r for k, (r, _) in _layer_shapes(case).items()}
        state["out"] = [{k: torch.empty(1, r, device=DEV) for k, r in rows.items() if k in ("q", "k", "v", "o", "down")}
                        for _ in range(case["layers"])]
        _layers(state)  # the first call loads the kernels
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            state["result"] = _layers(state)
        state["graph"] = graph
    return state


def _layers(state):
    case, lib, outs = state["case"], state["lib"], []
    q = getattr(tc_hip, case["type"])
    h, kv, ff = case["hidden"], case["kv"], case["ff"]
    for lay, o in zip(state["in"]["layers"], state["out"]):
        lib.gemv_multi(q, [lay["q"], lay["k"], lay["v"]], [lay["x"]] * 3, [h, kv, kv], [h, h, h], [o["q"], o["k"], o["v"]])
        lib.gemv(q, lay["o"], lay["attn"], h, h, out=o["o"])
        act, up = lib.gemv_dual(q, lay["gate"], lay["up"], lay["x2"], ff, h)
        lib.gemv(q, lay["down"], lay["h"], h, ff, out=o["down"])
        outs.append([o["q"], o["k"], o["v"], o["o"], act, up, o["down"]])
    return outs


def run(state):
    case, lib, a = state["case"], state["lib"], state["in"]
    op = case["op"]
    if op == "gemv":
        return lib.gemv(getattr(tc_hip, case["type"]), a["w"], a["x"], case["rows"], case["cols"])
    if op == "gemm":
        return lib.gemm(getattr(tc_hip, case["type"]), a["w"], a["x"], case["rows"], case["cols"])
    if op == "layer":
        state["graph"].replay()
        return state["result"]
    if op == "mixed":
        h, ff = case["hidden"], case["ff"]
        act, up = lib.gemv_dual(tc_hip.IQ3_XXS, a["gate"], a["up"], a["x"], ff, h)
        down = lib.gemv(tc_hip.Q6_K, a["down"], a["h"], h, ff)
        return [act, up, down, lib.gemv(tc_hip.Q6_K, a["head"], a["last"], case["vocab"], h)]
    if op == "moe":
        logits, ids, wts = lib.moe_router(a["router"], a["x"], case["K"])
        out = lib.moe_ffn(a["x"], ids, wts, a["gate"], a["up"], a["down"], case["E"], case["hidden"], case["ff"])
        return [logits, ids, wts, out]
    return lib.encode(getattr(tc_hip, case["type"]), a["x"])


# ---- what a pass cannot do without -------------------------------------------------


def _wbytes(t, rows, cols):
    return rows * tc_hip.row_bytes(getattr(tc_hip, t), cols)


def work(case):
    op = case["op"]
    if op in ("gemv", "gemm"):
        n, r, c = case["S"] if op == "gemv" else case["M"], case["rows"], case["cols"]
        return {"bytes": _wbytes(case["type"], r, c) + 4 * n * (r + c), "flops": 2 * n * r * c}
    if op == "layer":
        one = [(_wbytes(case["type"], r, c), r, c) for r, c in _layer_shapes(case).values()]
        x = 4 * (3 * case["hidden"] + case["ff"])  # q/k/v read one input, gate/up another
        return {"bytes": case["layers"] * (sum(w + 4 * r for w, r, _ in one) + x),
                "flops": case["layers"] * sum(2 * r * c for _, r, c in one)}
    if op == "mixed":
        h, ff, v = case["hidden"], case["ff"], case["vocab"]
        return {"bytes": 2 * _wbytes("IQ3_XXS", ff, h) + _wbytes("Q6_K", h, ff) + _wbytes("Q6_K", v, h) + 4 * (3 * h + 3 * ff + v),
                "flops": 2 * (3 * h * ff + h * v)}
    if op == "moe":
        T, E, K, H, F = case["T"], case["E"], case["K"], case["hidden"], case["ff"]
        used = E * (1 - (1 - K / E) ** T)  # experts that some token takes, for ids spread evenly
        expert = 2 * _wbytes("Q4_K", F, H) + _wbytes("Q4_K", H, F)
        return {"bytes": used * expert + 4 * (E * H + T * (2 * H + E + 2 * K)), "flops": 2 * T * H * E + 6 * T * K * H * F}
    r, c = case["rows"], case["cols"]
    return {"bytes": 4 * r * c + _wbytes(case["type"], r, c), "flops": 10 * r * c}


def tolerance(case):
    if case["op"] == "encode":
        return "exact"
    if case["op"] == "moe":
        # The hidden values are rounded to 8 bits between the products: sums in
        # another order move a few of them to the neighbouring step, max|h|/127,
        # which in the smallest block (1 token, 1 expert of 512) is 1.2e-3 of h.
        return {"rel": 3e-3, "max": 0.03, "differ": 0.0}
    # 32-bit sums of exact integer block products (or of fp32 activations):
    # 6e-8 to 1.6e-7 from the 64-bit results over the listed and drawn cases.
    return {"rel": 1e-6, "max": 2e-5}


# ---- the same results in 64 bits ----------------------------------------------------


def _grid(name, width):
    with open(os.path.join(GRID_DIR, name)) as f:
        text = re.sub(r"/\*.*?\*/", "", f.read(), flags=re.S)
    words = [int(v, 16) for v in re.findall(r"0x([0-9a-fA-F]+)", text)]
    return torch.tensor([[(v >> (8 * i)) & 255 for i in range(width)] for v in words], dtype=torch.int64, device=DEV)


def _half(b, off):
    return b[:, off:off + 2].contiguous().view(torch.float16).double()


def _bits(v, shifts, mask):
    return (v.unsqueeze(-1) >> torch.tensor(shifts, device=v.device)) & mask


def _nl(q):
    table = [-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113]
    return torch.tensor(table, dtype=torch.float64, device=q.device)[q]


def _signed7(idx):
    """Signs of 8 values from 7 bits and their parity."""
    bits = _bits(idx, range(7), 1)
    bits = torch.cat([bits, bits.sum(-1, keepdim=True) & 1], -1)
    return 1.0 - 2.0 * bits.double()


def _weights64(t, blocks):
    """Weights of raw blocks [n][block bytes] in 64 bits, [n][block values]."""
    b, n = blocks.to(torch.int64), blocks.shape[0]
    d = _half(blocks, SCALES[t][0][0])
    if t == "Q8_0":
        return d * blocks[:, 2:].contiguous().view(torch.int8).double()
    if t == "Q5_0":
        lo = torch.cat([b[:, 6:22] & 15, b[:, 6:22] >> 4], 1)
        return d * (lo + (_bits(b[:, 2:6], range(8), 1).view(n, 32) << 4) - 16).double()
    if t == "IQ4_NL":
        return d * _nl(torch.cat([b[:, 2:18] & 15, b[:, 2:18] >> 4], 1))
    if t in ("Q4_K", "Q5_K"):
        s = b[:, 4:16]
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
        qs = b[:, 16:] if t == "Q4_K" else b[:, 48:]
        q = _bits(qs.reshape(n, 4, 32), (0, 4), 15).permute(0, 1, 3, 2).reshape(n, 8, 32)
        if t == "Q5_K":
            q = q + (_bits(b[:, 16:48], range(8), 1).permute(0, 2, 1) << 4)
        dm = _half(blocks, 2)
        return ((d * sc.double()).unsqueeze(-1) * q.double() - (dm * mn.double()).unsqueeze(-1)).view(n, 256)
    if t == "Q2_K":
        q = _bits(b[:, 16:80].reshape(n, 2, 32), (0, 2, 4, 6), 3).permute(0, 1, 3, 2).reshape(n, 16, 16)
        sc, mn = b[:, 0:16] & 15, b[:, 0:16] >> 4
        return ((d * sc.double()).unsqueeze(-1) * q.double() - (_half(blocks, 82) * mn.double()).unsqueeze(-1)).view(n, 256)
    if t == "Q3_K":
        q = _bits(b[:, 32:96].reshape(n, 2, 32), (0, 2, 4, 6), 3).permute(0, 1, 3, 2).reshape(n, 8, 32)
        q = q - 4 * (1 - _bits(b[:, 0:32], range(8), 1).permute(0, 2, 1))
        s = b[:, 96:108]
        low = torch.cat([s[:, 0:8] & 15, s[:, 0:8] >> 4], 1)
        high = _bits(s[:, 8:12], (0, 2, 4, 6), 3).permute(0, 2, 1).reshape(n, 16)
        sc = (low | (high << 4)) - 32
        return ((d * sc.double()).unsqueeze(-1) * q.reshape(n, 16, 16).double()).view(n, 256)
    if t == "Q6_K":
        ql, qh = b[:, 0:128].reshape(n, 2, 2, 32), b[:, 128:192].reshape(n, 2, 32)
        lo = torch.cat([ql & 15, ql >> 4], 2)  # [n][half][quarter][32]
        q = (lo | (_bits(qh, (0, 2, 4, 6), 3).permute(0, 1, 3, 2) << 4)) - 32
        sc = blocks[:, 192:208].contiguous().view(torch.int8).double()
        return ((d * sc).unsqueeze(-1) * q.reshape(n, 16, 16).double()).view(n, 256)
    if t == "IQ4_XS":
        qs = b[:, 8:136].reshape(n, 8, 16)
        high = _bits(b[:, 2:4], (0, 2, 4, 6), 3).view(n, 8)
        low = _bits(b[:, 4:8], (0, 4), 15).view(n, 8)
        return ((d * (low + (high << 4) - 32).double()).unsqueeze(-1) * _nl(torch.cat([qs & 15, qs >> 4], 2))).view(n, 256)
    if t == "IQ3_XXS":
        g = _grid("iq3xxs_grid.inc", 4)[b[:, 2:66]].view(n, 8, 4, 8).double()
        aux = (b[:, 66:98].reshape(n, 8, 4) << torch.tensor([0, 8, 16, 24], device=DEV)).sum(-1)
        sign = _signed7(_bits(aux, (0, 7, 14, 21), 127))
        return ((d * (0.5 + (aux >> 28).double()) * 0.5).view(n, 8, 1, 1) * g * sign).view(n, 256)
    if t == "IQ3_S":
        idx = b[:, 2:66].reshape(n, 8, 8) | (_bits(b[:, 66:74], range(8), 1) << 8)
        g = _grid("iq3s_grid.inc", 4)[idx].view(n, 8, 4, 8).double()
        sign = 1.0 - 2.0 * _bits(b[:, 74:106].reshape(n, 8, 4), range(8), 1).double()
        return ((d * (1.0 + 2.0 * _bits(b[:, 106:110], (0, 4), 15).view(n, 8).double())).view(n, 8, 1, 1) * g * sign).view(n, 256)
    scales = _bits(b[:, 74:82] if t == "IQ2_S" else b[:, 66:74], (0, 4), 15).view(n, 8, 2).repeat_interleave(2, 2)
    if t == "IQ2_S":
        idx = b[:, 2:34].reshape(n, 8, 4) | (_bits(b[:, 66:74], (0, 2, 4, 6), 3) << 8)
        g = _grid("iq2s_grid.inc", 8)[idx].double()
        sign = 1.0 - 2.0 * _bits(b[:, 34:66].reshape(n, 8, 4), range(8), 1).double()
    else:
        q = (b[:, 2:66:2] | (b[:, 3:66:2] << 8)).view(n, 8, 4)
        g, sign = _grid("iq2xs_grid.inc", 8)[q & 511].double(), _signed7(q >> 9)
    return ((d.unsqueeze(-1) * (0.5 + scales.double()) * 0.25).unsqueeze(-1) * g * sign).view(n, 256)


def _act64(t, x):
    """The activations a product of type `t` works on: as they are, or rounded
    to 8 bits per block by the rule of the entry points (in 32 bits)."""
    if t in FP32_X:
        return x.double()
    blk = x.view(x.shape[0], -1, 32 if t == "Q8_0" else 256)
    top = blk.gather(-1, blk.abs().argmax(-1, keepdim=True)).double()
    inv = torch.where(top == 0, top, -127.0 / top).float().double()
    q = (inv * blk.double()).float().round().clamp(max=127.0)
    d = torch.where(inv == 0, inv, 1.0 / inv).float().double()
    return (d * q.double()).view(x.shape)


def _product64(t, w, x, rows, cols):
    """x @ W^T in 64 bits for activations x that are already what the product works on."""
    q = getattr(tc_hip, t)
    per = cols // tc_hip.BLOCK_SIZE[q]
    w = w.view(rows, per, tc_hip.TYPE_SIZE[q])
    out = torch.empty(x.shape[0], rows, dtype=torch.float64, device=DEV)
    step = max(1, 2 ** 24 // cols)
    for r in range(0, rows, step):
        part = w[r:r + step]
        out[:, r:r + step] = x @ _weights64(t, part.reshape(-1, tc_hip.TYPE_SIZE[q])).view(part.shape[0], cols).t()
    return out


def _pair64(t, gate, up, x, rows, cols):
    u = _product64(t, up, x, rows, cols)
    return torch.nn.functional.silu(_product64(t, gate, x, rows, cols)) * u, u


def exact(case, seed):
    op = case["op"]
    if op == "encode":
        return None  # bytes
    a = _inputs(case, seed)
    if op in ("gemv", "gemm"):
        return _product64(case["type"], a["w"], _act64(case["type"], a["x"]), case["rows"], case["cols"])
    if op == "layer":
        t, sh, outs = case["type"], _layer_shapes(case), []
        for lay in a["layers"]:
            x, one = _act64(t, lay["x"]), []
            one += [_product64(t, lay[k], x, *sh[k]) for k in ("q", "k", "v")]
            one.append(_product64(t, lay["o"], _act64(t, lay["attn"]), *sh["o"]))
            one += [v.view(-1) for v in _pair64(t, lay["gate"], lay["up"], _act64(t, lay["x2"]), *sh["gate"])]
            one.append(_product64(t, lay["down"], _act64(t, lay["h"]), *sh["down"]))
            outs.append(one)
        return outs
    if op == "mixed":
        h, ff = case["hidden"], case["ff"]
        act, up = _pair64("IQ3_XXS", a["gate"], a["up"], _act64("IQ3_XXS", a["x"]), ff, h)
        return [act.view(-1), up.view(-1), _product64("Q6_K", a["down"], _act64("Q6_K", a["h"]), h, ff),
                _product64("Q6_K", a["head"], _act64("Q6_K", a["last"]), case["vocab"], h)]
    # moe: the hidden values are kept in 64 bits here (the path rounds them to 8)
    E, H, F, K = case["E"], case["hidden"], case["ff"], case["K"]
    logits = a["x"].double() @ a["router"].double().t()
    wts, ids = torch.softmax(logits, -1).topk(K, -1)
    wts = wts / wts.sum(-1, keepdim=True)
    x, out = _act64("Q4_K", a["x"]), torch.zeros(case["T"], H, dtype=torch.float64, device=DEV)
    per = {k: a[k].view(E, -1) for k in ("gate", "up", "down")}
    for e in range(E):
        tok, rank = (ids == e).nonzero(as_tuple=True)
        if len(tok):
            hid, _ = _pair64("Q4_K", per["gate"][e], per["up"][e], x[tok], F, H)
            out.index_add_(0, tok, wts[tok, rank].unsqueeze(1) * _product64("Q4_K", per["down"][e], hid, H, F))
    return [logits, None, wts, out]
