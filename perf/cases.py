"""Performance cases of the fused layer ops: the work a model's forward pass hands to this provider.

Every case goes through a public entry point (``sharplight_amd.native``'s ops on device pointers, or a compiled
segment of ``sharplight_amd.provider`` on host arrays). Inputs live in torch tensors made on the GPU from the seed;
outputs are the caller's own preallocated tensors, as in a serving loop. ``exact`` restates each op in 64-bit torch.

Ranges that ``draw`` covers: row norms, gated activations, rope, table gathers and fused groups from one token to a
long prefill, and matrix products with [N, K] weights (one matrix, or a gate/up pair with the SiLU epilogue) from one
token (decode) over a batch of sequences to a 512-token prefill, float activations and integer-dot numerics, in the
weight formats of Q4_K_M / Q8_0 / Q4_0 files and of unquantized checkpoints.
"""
import math

import numpy as np
import torch

from sharplight_amd import native, provider

DEV = "cuda"
TORCH = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
SIZE = {"f32": 4, "bf16": 2, "f16": 2}
# values and bytes per block of the quantized formats
BLOCK = {"q8_0": (32, 34), "q4_0": (32, 18), "q4_k": (256, 144), "q5_k": (256, 176), "q6_k": (256, 210)}
EPS = 1e-6


def listed():
    return [
        # the smallest call: a 0.6B model's RMSNorm over a short prompt, where launch and latency are most of it
        {"name": "norm_small", "op": "norm", "kind": "rms", "rows": 512, "dim": 1024, "dtype": "f32", "residual": False},
        # the norm before every attention and FFN block of an 8B model in a long prefill: residual add + RMSNorm
        {"name": "add_norm_prefill", "op": "norm", "kind": "rms", "rows": 8192, "dim": 4096, "dtype": "bf16", "residual": True},
        # the FFN's gated activation in the same prefill (the largest by bytes)
        {"name": "swiglu_prefill", "op": "gated", "act": "silu", "rows": 8192, "cols": 14336, "dtype": "bf16", "merged": False},
        # the attention prologue: per-head q/k RMSNorm + neox rope, k straight into a paged KV cache
        {"name": "qk_rope_prefill", "op": "rope", "tokens": 4096, "heads": 32, "kv_heads": 8, "head_dim": 128, "neox": True,
         "norm": True, "paged": True},
        # token embedding of a prefill from a Q4_K table
        {"name": "gather_q4_k", "op": "gather", "fmt": "q4_k", "vocab": 151936, "dim": 4096, "ids": 16384},
        # bias add + residual add + RMSNorm as one fused group (f32 graphs with biased projections)
        {"name": "group_norm_prefill", "op": "group", "rows": 8192, "cols": 4096},
        # one decode step's gate/up projections, the default numerics (activations quantized, integer dots)
        {"name": "ffn_token_q4_k", "op": "linear", "fmt": "q4_k", "tokens": 1, "k": 4096, "n": 14336, "pair": True, "x": "f32", "int8": True},
        # the same for a batch of sequences
        {"name": "ffn_batch_q4_k", "op": "linear", "fmt": "q4_k", "tokens": 16, "k": 4096, "n": 14336, "pair": True, "x": "f32", "int8": True},
        # a small batch's down projection with float activations (a MatMul marked f32_activations; Q6_K in Q4_K_M files)
        {"name": "down_batch_q6_k", "op": "linear", "fmt": "q6_k", "tokens": 6, "k": 14336, "n": 4096, "pair": False, "x": "f32", "int8": False},
        # a 512-token prompt's gate/up projections on quantized weights
        {"name": "ffn_prefill_q4_k", "op": "linear", "fmt": "q4_k", "tokens": 512, "k": 4096, "n": 14336, "pair": True, "x": "f32", "int8": False},
        # an unquantized model's projection in a prefill of ragged length, K off the power-of-two grid
        {"name": "proj_prefill_bf16", "op": "linear", "fmt": "bf16", "tokens": 331, "k": 2880, "n": 4096, "pair": False, "x": "bf16", "int8": False},
        # a whole call: one decode step of an FFN half-layer (norm, gate/up, activation, down, residual) as a compiled segment
        {"name": "segment_ffn_token", "op": "segment", "fmt": "q4_k", "tokens": 1, "hidden": 4096, "ffn": 14336},
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(["norm", "gated", "rope", "gather", "group", "segment"] + ["linear"] * 6)
    if op == "norm":
        kind = rng.choice(["rms", "rms", "layer"])
        return {"op": op, "kind": kind, "rows": _log(rng, 1, 8192), "dim": 8 * _log(rng, 64, 1024),
                "dtype": rng.choice(["f32", "bf16"]), "residual": kind == "rms" and rng.random() < 0.5}
    if op == "gated":
        return {"op": op, "act": rng.choice(["silu", "gelu_tanh", "gelu_erf"]), "rows": _log(rng, 1, 4096),
                "cols": 8 * _log(rng, 128, 2048), "dtype": rng.choice(["f32", "bf16"]), "merged": rng.random() < 0.5}
    if op == "rope":
        kv = rng.choice([1, 2, 4, 8])
        return {"op": op, "tokens": _log(rng, 1, 8192), "heads": kv * rng.choice([2, 4, 5, 8]), "kv_heads": kv,
                "head_dim": rng.choice([64, 128, 256]), "neox": rng.random() < 0.7, "norm": rng.random() < 0.5,
                "paged": rng.random() < 0.5}
    if op == "gather":
        return {"op": op, "fmt": rng.choice(["q8_0", "q4_0", "q4_k", "q6_k", "bf16"]), "vocab": rng.randint(32000, 151936),
                "dim": 256 * rng.randint(4, 20), "ids": _log(rng, 1, 16384)}
    if op == "group":
        return {"op": op, "rows": _log(rng, 1, 8192), "cols": 8 * _log(rng, 64, 640)}
    if op == "segment":
        return {"op": op, "fmt": rng.choice(["q8_0", "q4_k", "q5_k"]), "tokens": _log(rng, 1, 128),
                "hidden": 256 * rng.randint(4, 16), "ffn": 256 * rng.randint(16, 48)}
    fmt = rng.choice(["q4_k", "q4_k", "q6_k", "q5_k", "q8_0", "q4_0", "bf16", "f16"])
    quant = fmt in BLOCK
    c = {"op": op, "fmt": fmt, "tokens": _log(rng, 1, 512), "k": 256 * rng.randint(4, 56) if quant else 64 * rng.randint(16, 256),
         "n": _log(rng, 500, 16384), "pair": rng.random() < 0.5, "x": rng.choice(["f32", "f32", "bf16"]),
         "int8": quant and rng.random() < 0.5}
    if c["int8"]:  # the integer-dot rule takes 1..31 rows
        c["tokens"] = _log(rng, 1, 31)
    # no costlier than the largest listed case (a value of an unquantized matrix is read at full width)
    most = 512 * 4096 * 14336 * 2 // (1 if quant else 4)
    while c["tokens"] * c["k"] * c["n"] * (2 if c["pair"] else 1) > most:
        c["n"] = c["n"] // 2 + 1
    return c


# ---- inputs -----------------------------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _normal(g, shape, dtype="f32", mean=0.0, std=1.0):
    return torch.randn(shape, generator=g, device=DEV).mul_(std).add_(mean).to(TORCH[dtype])


def _uniform(g, shape, lo, hi):
    return torch.rand(shape, generator=g, device=DEV).mul_(hi - lo).add_(lo)


def _half_bytes(v):
    return v.to(torch.float16).unsqueeze(-1).view(torch.uint8)


def _table(g, fmt, rows, dim):
    """Weights [rows, dim] in fmt: random codes, block scales that give values of about 0.02 to 0.04 (a trained matrix's)."""
    if fmt in TORCH:
        return _normal(g, (rows, dim), fmt, std=0.02)
    bs, bb = BLOCK[fmt]
    t = torch.randint(0, 256, (rows, dim // bs, bb), generator=g, device=DEV, dtype=torch.uint8)
    d = lambda lo, hi: _uniform(g, (rows, dim // bs), lo, hi)
    if fmt == "q8_0":
        t[:, :, 0:2] = _half_bytes(d(1e-4, 5e-4))
    elif fmt == "q4_0":
        t[:, :, 0:2] = _half_bytes(d(2e-3, 6e-3))
    elif fmt == "q6_k":
        t[:, :, 208:210] = _half_bytes(d(1e-5, 4e-5))
    else:  # the block minimum of about the codes' middle
        s = d(1e-4, 4e-4) if fmt == "q4_k" else d(5e-5, 2e-4)
        t[:, :, 0:2] = _half_bytes(s)
        t[:, :, 2:4] = _half_bytes(s * (7.5 if fmt == "q4_k" else 15.5))
    return t.reshape(rows, -1)


def prepare(case, seed):
    g = _gen(seed)
    s = {"case": case}
    return globals()["_prepare_" + case["op"]](s, g, **{k: v for k, v in case.items() if k not in ("name", "op")})


def _prepare_norm(s, g, kind, rows, dim, dtype, residual):
    s["x"] = _normal(g, (rows, dim), dtype)
    s["res"] = _normal(g, (rows, dim), dtype) if residual else None
    s["w"] = _normal(g, (dim,), mean=1.0, std=0.1)
    s["b"] = _normal(g, (dim,), std=0.1) if kind == "layer" else None
    s["y"] = torch.empty_like(s["x"])
    s["h"] = torch.empty_like(s["x"]) if residual else None
    return s


def _prepare_gated(s, g, act, rows, cols, dtype, merged):
    if merged:  # one projection's output, gate and up side by side
        m = _normal(g, (rows, 2 * cols), dtype)
        s["gate"], s["up"], s["stride"] = m[:, :cols], m[:, cols:], 2 * cols
    else:
        s["gate"], s["up"], s["stride"] = _normal(g, (rows, cols), dtype), _normal(g, (rows, cols), dtype), cols
    s["out"] = torch.empty((rows, cols), dtype=TORCH[dtype], device=DEV)
    return s


CTX, PAGE = 32768, 16  # the KV cache's rows and block size


def _prepare_rope(s, g, tokens, heads, kv_heads, head_dim, neox, norm, paged):
    s["q"] = _normal(g, (tokens, heads, head_dim), "bf16")
    s["k"] = _normal(g, (tokens, kv_heads, head_dim), "bf16")
    s["wq"] = _normal(g, (head_dim,), mean=1.0, std=0.1) if norm else None
    s["wk"] = _normal(g, (head_dim,), mean=1.0, std=0.1) if norm else None
    pos = torch.randperm(CTX, generator=g, device=DEV)[:tokens].sort().values.to(torch.int32)
    s["pos"], s["yq"] = pos, torch.empty_like(s["q"])
    s["rows"] = None
    if paged:  # one sequence; its blocks anywhere in the cache
        s["seq"] = torch.zeros((tokens, 4), dtype=torch.int32, device=DEV)
        s["seq"][:, 1] = pos
        s["pages"] = torch.randperm(CTX // PAGE, generator=g, device=DEV).to(torch.int32)
        s["yk"] = torch.zeros((CTX, kv_heads, head_dim), dtype=torch.bfloat16, device=DEV)
        s["rows"] = native.cache_rows("paged", CTX, seq=s["seq"].data_ptr(), pages=s["pages"].data_ptr(), page_slots=1,
                                      blocks_per_slot=CTX // PAGE, block_size=PAGE)
    else:
        s["yk"] = torch.empty_like(s["k"])
    return s


def _prepare_gather(s, g, fmt, vocab, dim, ids):
    s["table"] = _table(g, fmt, vocab, dim)
    s["ids"] = torch.randint(0, vocab, (ids,), generator=g, device=DEV, dtype=torch.int32)
    s["y"] = torch.empty((ids, dim), dtype=torch.bfloat16, device=DEV)
    return s


def _prepare_group(s, g, rows, cols):
    s["x"], s["res"] = _normal(g, (rows, cols)), _normal(g, (rows, cols))
    s["bias"], s["w"] = _normal(g, (cols,)), _normal(g, (cols,), mean=1.0, std=0.1)
    s["h"], s["y"] = torch.empty_like(s["x"]), torch.empty_like(s["x"])
    return s


def _prepare_linear(s, g, fmt, tokens, k, n, pair, x, int8):
    s["x"] = _normal(g, (tokens, k), x)
    s["w"] = _table(g, fmt, n, k)
    s["w2"] = _table(g, fmt, n, k) if pair else None
    s["y"] = torch.empty((tokens, n), dtype=TORCH[x], device=DEV)
    s["xq"] = torch.empty(tokens * native.q8_row_bytes(k), dtype=torch.uint8, device=DEV) if int8 else None
    return s


def _inputs_segment(s, g, fmt, tokens, hidden, ffn):
    s["x"] = _normal(g, (tokens, hidden))
    s["w"] = _normal(g, (hidden,), mean=1.0, std=0.1)
    s["gate"], s["up"], s["down"] = _table(g, fmt, ffn, hidden), _table(g, fmt, ffn, hidden), _table(g, fmt, hidden, ffn)
    return s


def _prepare_segment(s, g, fmt, tokens, hidden, ffn):
    _inputs_segment(s, g, fmt, tokens, hidden, ffn)
    b = provider.GraphBuilder()
    x = b.input("f32", "T", hidden)
    w, wg, wu, wd = b.weight("f32", hidden), b.weight(fmt, ffn, hidden), b.weight(fmt, ffn, hidden), b.weight(fmt, hidden, ffn)
    n = b.rms_norm(x, w, EPS)
    a = b.mul(b.silu(b.matmul(n, wg)), b.matmul(n, wu))
    y = b.output(b.add(x, b.matmul(a, wd)))
    p = provider.HipExecutionProvider()
    seg = p.open_device(p.get_devices()[0]).compile(b, max_tokens=max(tokens, 16))
    for v, t in ((w, s["w"]), (wg, s["gate"]), (wu, s["up"]), (wd, s["down"])):
        seg.set_input(v, t.cpu().numpy())
    s["host"], s["in"], s["out"], s["seg"] = s["x"].cpu().numpy(), x, y, seg
    return s


# ---- one pass ---------------------------------------------------------------------------------------------

def _p(t):
    return None if t is None else t.data_ptr()


def run(s):
    return globals()["_run_" + s["case"]["op"]](s, s["case"])


def _run_norm(s, c):
    native.rownorm(c["kind"], c["dtype"], c["dtype"], _p(s["x"]), _p(s["y"]), c["rows"], c["dim"], res=_p(s["res"]),
                   w=_p(s["w"]), b=_p(s["b"]), h_out=_p(s["h"]), eps=EPS)
    return [s["y"], s["h"]] if c["residual"] else [s["y"]]


def _run_gated(s, c):
    native.gated_act(c["act"], c["dtype"], c["dtype"], _p(s["gate"]), _p(s["up"]), _p(s["out"]), c["rows"], c["cols"],
                     gate_stride=s["stride"], up_stride=s["stride"])
    return s["out"]


def _run_rope(s, c):
    q = {"x": _p(s["q"]), "y": _p(s["yq"]), "heads": c["heads"], "norm_w": _p(s["wq"])}
    k = {"x": _p(s["k"]), "y": _p(s["yk"]), "heads": c["kv_heads"], "norm_w": _p(s["wk"])}
    if s["rows"] is not None:
        k["rows"] = s["rows"]
    native.rope("bf16", "bf16", [q, k], _p(s["pos"]), c["tokens"], c["head_dim"], neox=c["neox"], base=1e6, norm=c["norm"],
                eps=EPS)
    return [s["yq"], s["yk"]]


def _run_gather(s, c):
    native.gather(c["fmt"], _p(s["table"]), c["vocab"], c["dim"], _p(s["ids"]), c["ids"], "bf16", _p(s["y"]))
    return s["y"]


def _run_group(s, c):
    native.ew_program([(_p(s["x"]), "f32", native.EWI_FULL), (_p(s["bias"]), "f32", native.EWI_ROW),
                       (_p(s["res"]), "f32", native.EWI_FULL)],
                      [("binary", "Add", 0, 1, 3, "f32", 0, 0), ("binary", "Add", 3, 2, 3, "f32", 0, 0)],
                      [(_p(s["h"]), "f32", 3)], c["rows"], c["cols"],
                      tail={"kind": "rms", "reg": 3, "w": _p(s["w"]), "eps": EPS, "y": _p(s["y"]), "dtype_y": "f32"})
    return [s["h"], s["y"]]


def _run_linear(s, c):
    T, K, N, f, xt = c["tokens"], c["k"], c["n"], c["fmt"], c["x"]
    if c["int8"]:
        native.quantize_q8(xt, _p(s["x"]), T, K, _p(s["xq"]))
        if c["pair"]:
            native.dual_matvec_q8("silu", f, xt, _p(s["xq"]), T, K, _p(s["w"]), _p(s["w2"]), N, _p(s["y"]))
        else:
            native.matvec_q8(f, xt, _p(s["xq"]), T, K, _p(s["w"]), N, _p(s["y"]))
    elif c["pair"]:
        native.dual_matvec("silu", f, xt, xt, _p(s["x"]), T, K, _p(s["w"]), _p(s["w2"]), N, _p(s["y"]))
    else:
        native.matvec(f, xt, xt, _p(s["x"]), T, K, _p(s["w"]), N, _p(s["y"]))
    return s["y"]


def _run_segment(s, c):
    seg = s["seg"]
    seg.set_input(s["in"], s["host"])
    seg.execute(c["tokens"])
    return seg.get_output(s["out"])


# ---- what a pass cannot do without ---------------------------------------------------------------------------

def _weight_bytes(fmt, n):
    return n * SIZE[fmt] if fmt in SIZE else n // BLOCK[fmt][0] * BLOCK[fmt][1]


def work(case):
    c = case
    if c["op"] == "norm":
        n = c["rows"] * c["dim"]
        return {"bytes": n * SIZE[c["dtype"]] * (4 if c["residual"] else 2) + c["dim"] * 4, "flops": 5 * n}
    if c["op"] == "gated":
        n = c["rows"] * c["cols"]
        return {"bytes": 3 * n * SIZE[c["dtype"]], "flops": 8 * n}
    if c["op"] == "rope":
        n = c["tokens"] * (c["heads"] + c["kv_heads"]) * c["head_dim"]
        return {"bytes": 4 * n + 4 * c["tokens"], "flops": 6 * n}
    if c["op"] == "gather":
        return {"bytes": c["ids"] * (_weight_bytes(c["fmt"], c["dim"]) + 4 + 2 * c["dim"]), "flops": 2 * c["ids"] * c["dim"]}
    if c["op"] == "group":
        n = c["rows"] * c["cols"]
        return {"bytes": 16 * n + 8 * c["cols"], "flops": 6 * n}
    if c["op"] == "segment":
        n = 3 * c["hidden"] * c["ffn"]
        return {"bytes": _weight_bytes(c["fmt"], n) + 8 * c["tokens"] * c["hidden"], "flops": 2 * n * c["tokens"]}
    n = c["k"] * c["n"] * (2 if c["pair"] else 1)
    return {"bytes": _weight_bytes(c["fmt"], n) + SIZE[c["x"]] * c["tokens"] * (c["k"] + c["n"]), "flops": 2 * n * c["tokens"]}


def tolerance(case):
    c = case
    if c["op"] == "gather":
        return "exact"  # dequantization is bit for bit
    bf16 = c.get("dtype") == "bf16" or c.get("x") == "bf16" or c["op"] == "rope"
    if bf16:  # another order of f32 sums moves a few values over a rounding boundary (2^-8 of the value each)
        return {"rel": 2e-3, "max": 2e-2}
    if c["op"] == "segment":  # a last-bit change before the quantizer moves a few int8 codes
        return {"rel": 2e-4, "max": 5e-3}
    if c["op"] == "linear":  # f32 sums of up to 16384 terms in another order (2e-7 to 4e-7 from the exact result)
        return {"rel": 2e-6, "max": 1e-4}
    return {"rel": 5e-7, "max": 2e-5}


# ---- 64-bit reference ---------------------------------------------------------------------------------------

def _half(t):
    return t.contiguous().view(torch.float16).double()  # [..., 2] bytes -> [..., 1]


def _decode(fmt, t, rows, dim):
    """Weights [rows, dim] of raw blocks in 64 bits (ggml's block layouts)."""
    if fmt in TORCH:
        return t.double()
    bs, bb = BLOCK[fmt]
    t = t.reshape(rows, dim // bs, bb)
    if fmt == "q8_0":
        v = t[..., 2:].contiguous().view(torch.int8).double() * _half(t[..., :2])
    elif fmt == "q4_0":
        q = t[..., 2:]
        v = (torch.cat([q & 15, q >> 4], -1).double() - 8) * _half(t[..., :2])
    elif fmt == "q6_k":
        out = []
        for h in range(2):
            ql, qh = t[..., 64 * h:64 * h + 64], t[..., 128 + 32 * h:160 + 32 * h]
            for k in range(4):
                lo = ql[..., 32 * (k & 1):32 * (k & 1) + 32]
                lo = lo >> 4 if k >= 2 else lo & 15
                q = (lo | (((qh >> (2 * k)) & 3) << 4)).double() - 32
                sc = t[..., 192 + 8 * h + 2 * k:194 + 8 * h + 2 * k].contiguous().view(torch.int8).double()
                out.append(q * sc.repeat_interleave(16, -1))
        v = torch.cat(out, -1) * _half(t[..., 208:210])
    else:  # q4_k, q5_k
        d, m, s = _half(t[..., 0:2]), _half(t[..., 2:4]), t[..., 4:16]
        out = []
        for j in range(8):
            if j < 4:
                sc, mn = s[..., j] & 63, s[..., j + 4] & 63
            else:
                sc = (s[..., j + 4] & 15) | ((s[..., j - 4] >> 6) << 4)
                mn = (s[..., j + 4] >> 4) | ((s[..., j] >> 6) << 4)
            o = (16 if fmt == "q4_k" else 48) + 32 * (j // 2)
            q = t[..., o:o + 32]
            q = q >> 4 if j & 1 else q & 15
            if fmt == "q5_k":
                q = q | (((t[..., 16:48] >> j) & 1) << 4)
            out.append(q.double() * (d * sc.unsqueeze(-1).double()) - m * mn.unsqueeze(-1).double())
        v = torch.cat(out, -1)
    return v.reshape(rows, dim)


def _q8(x):
    """The integer-dot numerics' activations: int8 codes per 32 values with a 32-bit scale, as 64-bit values."""
    x = x.float()
    b = x.reshape(x.shape[0], -1, 32)
    d = b.abs().amax(-1, keepdim=True) / 127.0
    inv = torch.where(d > 0, 1.0 / d, torch.zeros_like(d))
    p = b * inv
    q = (p + torch.copysign(torch.full_like(p, 0.5), p)).trunc()
    return (q.double() * d.double()).reshape(x.shape)


def _product(x, fmt, w, n, k):
    """x . W^T in 64 bits, a slice of the rows at a time (the decoded weights of a large matrix take gigabytes)."""
    step = max(1, (1 << 26) // k)
    return torch.cat([x @ _decode(fmt, w[i:i + step], min(step, n - i), k).T for i in range(0, n, step)], 1)


def _silu(v):
    return v * torch.sigmoid(v)


def exact(case, seed):
    make = _inputs_segment if case["op"] == "segment" else globals()["_prepare_" + case["op"]]
    s = make({"case": case}, _gen(seed), **{k: v for k, v in case.items() if k not in ("name", "op")})
    c = case
    if c["op"] == "norm":
        x = s["x"].double() + (s["res"].double() if c["residual"] else 0)
        if c["kind"] == "layer":
            v = x - x.mean(-1, keepdim=True)
            y = v * torch.rsqrt(v.square().mean(-1, keepdim=True) + EPS) * s["w"].double() + s["b"].double()
        else:
            y = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * s["w"].double()
        return [y, x] if c["residual"] else [y]
    if c["op"] == "gated":
        step = max(1, (1 << 26) // c["cols"])
        out = []
        for i in range(0, c["rows"], step):
            g, u = s["gate"][i:i + step].double(), s["up"][i:i + step].double()
            if c["act"] == "silu":
                a = _silu(g)
            else:
                a = torch.nn.functional.gelu(g, approximate="tanh" if c["act"] == "gelu_tanh" else "none")
            out.append(a * u)
        return torch.cat(out)
    if c["op"] == "rope":
        D = c["head_dim"]
        inv = 1e6 ** (-2.0 * torch.arange(D // 2, device=DEV, dtype=torch.float64) / D)
        ang = s["pos"].double()[:, None, None] * inv
        out = []
        for x, w in ((s["q"], s["wq"]), (s["k"], s["wk"])):
            x = x.double()
            if c["norm"]:
                x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()
            a, b = (x[..., :D // 2], x[..., D // 2:]) if c["neox"] else (x[..., 0::2], x[..., 1::2])
            a, b = a * ang.cos() - b * ang.sin(), a * ang.sin() + b * ang.cos()
            out.append(torch.cat([a, b], -1) if c["neox"] else torch.stack([a, b], -1).reshape(x.shape))
        if c["paged"]:
            pos = s["pos"].long()
            cache = torch.zeros(s["yk"].shape, dtype=torch.float64, device=DEV)
            cache[s["pages"].long()[pos // PAGE] * PAGE + pos % PAGE] = out[1]
            out[1] = cache
        return out
    if c["op"] == "gather":
        return _decode(c["fmt"], s["table"][s["ids"].long()], c["ids"], c["dim"])
    if c["op"] == "group":
        h = s["x"].double() + s["bias"].double() + s["res"].double()
        return [h, h * torch.rsqrt(h.square().mean(-1, keepdim=True) + EPS) * s["w"].double()]
    if c["op"] == "segment":
        # the default rule: Q8_0 takes integer dots from 2 to 16 rows, the K-quants from 1 to 8
        int8 = 2 <= c["tokens"] <= 16 if c["fmt"] == "q8_0" else c["tokens"] <= 8
        q = _q8 if int8 else (lambda v: v.double())
        x, h, f = s["x"].double(), c["hidden"], c["ffn"]
        n = q(x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * s["w"].double())
        a = _silu(_product(n, c["fmt"], s["gate"], f, h)) * _product(n, c["fmt"], s["up"], f, h)
        return (x + _product(q(a), c["fmt"], s["down"], h, f)).cpu().numpy()
    x = _q8(s["x"]) if c["int8"] else s["x"].double()
    y = _product(x, c["fmt"], s["w"], c["n"], c["k"])
    return _silu(y) * _product(x, c["fmt"], s["w2"], c["n"], c["k"]) if c["pair"] else y
