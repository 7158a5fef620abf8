"""Performance cases of the GEMM, attention and tile-op path.

A case is one call as a user's program makes it: a GEMM or an attention
forward through `frisk_amd.runtime` (the binding of the C-ABI), a GEMM
program of the tile IR through `frisk_amd.execute`, or a tile op (reduce,
copy, fill).  `listed()` holds fixed cases, `draw()` gives more of the same
ranges, odd sizes among them.

Fields of a case (all plain values):
  op "gemm":   m, n, k, dtype ("bf16", "f16", "f32", "fp8", "int8"), out,
               layout ("nt": A [M, K], B [N, K]; "nn", "tn", "tt" likewise),
               accumulate (C += A.B), via ("runtime" or "execute")
  op "attn":   batch, heads, seq_q, seq_k, head_dim, dtype, out, causal,
               lse, layout ("bhsd", or "bshd": heads interleaved),
               k_transposed (K stored [batch, heads, head_dim, seq_k])
  op "reduce": rows, cols, axis, kind, dtype
  op "copy":   rows, cols, dtype, out, padded (rows of a wider buffer)
  op "fill":   rows, cols, dtype
"""
import math

import torch

import frisk_amd as F
from frisk_amd import runtime as rt

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32,
          "fp8": torch.float8_e4m3fn, "int8": torch.int8, "int32": torch.int32}
BYTES = {"bf16": 2, "f16": 2, "f32": 4, "fp8": 1, "int8": 1, "int32": 4}
# Names of the element types in the IR builder.
IR_NAMES = {"bf16": "bf16", "f16": "fp16", "f32": "fp32", "fp8": "e4m3fn", "int8": "int8",
            "int32": "int32"}


def _gemm(name, m, n, k, dtype, out, layout, accumulate=False, via="runtime"):
    return {"name": name, "op": "gemm", "m": m, "n": n, "k": k, "dtype": dtype, "out": out,
            "layout": layout, "accumulate": accumulate, "via": via}


def _attn(name, batch, heads, seq_q, seq_k, head_dim, dtype, out, causal, lse=False,
          layout="bhsd", k_transposed=False):
    return {"name": name, "op": "attn", "batch": batch, "heads": heads, "seq_q": seq_q,
            "seq_k": seq_k, "head_dim": head_dim, "dtype": dtype, "out": out, "causal": causal,
            "lse": lse, "layout": layout, "k_transposed": k_transposed}


def listed():
    return [
        # One decode step of a projection: 16 tokens against a square weight.
        _gemm("gemm_decode_bf16", 16, 4096, 4096, "bf16", "bf16", "nt"),
        # The same step with quantised weights and activations: the weight of
        # the quantised GEMM below.
        _gemm("gemm_decode_fp8", 32, 8192, 8192, "fp8", "bf16", "nt"),
        # A large decode batch through the widest projection, in the storage
        # order the IR builder defaults to (neither operand transposed).
        _gemm("gemm_batch128_bf16_nn", 128, 14336, 4096, "bf16", "bf16", "nn"),
        # A prefill chunk of 1024 tokens through a square projection.
        _gemm("gemm_chunk1024_bf16", 1024, 4096, 4096, "bf16", "bf16", "nt"),
        # The headline training / prefill GEMM.
        _gemm("gemm_bf16_4096", 4096, 4096, 4096, "bf16", "bf16", "nt"),
        # The quantised GEMM with per-tensor scales.
        _gemm("gemm_fp8_4096x8192x8192", 4096, 8192, 8192, "fp8", "bf16", "nt"),
        # Odd, ragged sizes: rows that do not start on 16-byte boundaries.
        _gemm("gemm_ragged_f16", 1111, 3333, 1777, "f16", "f16", "nt"),
        # The small fp32 program of the IR builder, run as a program: the
        # latency of recognising it and launching its kernel counts.
        _gemm("execute_f32_512_nn", 512, 512, 512, "f32", "f32", "nn", via="execute"),
        # Prefill attention of a whole batch: the largest case.
        _attn("attn_prefill_causal", 4, 32, 4096, 4096, 128, "bf16", "bf16", True),
        # A short ragged sequence at head_dim 64, f32 output.
        _attn("attn_s1025_d64", 2, 32, 1025, 1025, 64, "f16", "f32", False),
        # One decode step of attention over a filled KV cache.
        _attn("attn_decode", 4, 32, 1, 4096, 128, "bf16", "bf16", True),
        # Column statistics of a large activation.
        {"name": "reduce_max_cols", "op": "reduce", "rows": 8192, "cols": 16384, "axis": 0,
         "kind": "max", "dtype": "f32"},
    ]


def _log(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return int(min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _size(rng, lo, hi):
    """Half multiples of 128, a quarter multiples of 8, a quarter any number."""
    x, kind = _log(rng, lo, hi), rng.random()
    step = 128 if kind < 0.5 else 8 if kind < 0.75 else 1
    return max(step, x // step * step)


def _draw_gemm(rng):
    dtype = rng.choice(["bf16", "bf16", "f16", "f32", "fp8", "int8"])
    out = {"bf16": rng.choice(["bf16", "bf16", "f32"]), "f16": rng.choice(["f16", "f16", "f32"]),
           "f32": "f32", "fp8": rng.choice(["bf16", "bf16", "f16", "f32"]), "int8": "int32"}[dtype]
    layout = rng.choice(["nt", "nt", "nt", "nn", "nn", "tn", "tt"])
    # f32 runs at a sixteenth of the matrix rate: a smaller range.
    top = 2e10 if dtype == "f32" else 1.5e11
    while True:
        m = rng.choice([_log(rng, 1, 128), _size(rng, 128, 8192)])
        n, k = _size(rng, 64, 14336), _size(rng, 64, 14336)
        if 2.0 * m * n * k <= top and m * n * k >= 1 << 22:
            break
    return {"op": "gemm", "m": m, "n": n, "k": k, "dtype": dtype, "out": out, "layout": layout,
            "accumulate": rng.random() < 0.1, "via": "execute" if rng.random() < 0.15 else "runtime"}


def _draw_attn(rng):
    head_dim = rng.choice([128, 128, 128, 64, 64, 32, 16])
    dtype = rng.choice(["bf16", "bf16", "f16"])
    decode = rng.random() < 0.45
    while True:
        batch, heads = _log(rng, 1, 64), rng.choice([1, 4, 8, 16, 32, 32])
        if decode:
            seq_q, seq_k = rng.choice([1, 1, 1, _log(rng, 2, 16)]), _size(rng, 64, 32768)
        else:
            seq_q = seq_k = _size(rng, 64, 8192)
        flops = 4.0 * batch * heads * seq_q * seq_k * head_dim
        kv = 4.0 * batch * heads * seq_k * head_dim
        if flops <= 2.5e11 and kv <= 6e8 and seq_q <= seq_k:
            break
    k_transposed = seq_k % 8 == 0 and rng.random() < 0.1
    return {"op": "attn", "batch": batch, "heads": heads, "seq_q": seq_q, "seq_k": seq_k,
            "head_dim": head_dim, "dtype": dtype, "out": "f32" if rng.random() < 0.2 else dtype,
            "causal": rng.random() < 0.6, "lse": rng.random() < 0.3,
            "layout": rng.choice(["bhsd", "bshd"]), "k_transposed": k_transposed}


def _draw_tile(rng):
    op = rng.choice(["reduce", "reduce", "copy", "fill"])
    while True:
        rows, cols = _size(rng, 16, 32768), _size(rng, 16, 32768)
        if 1 << 16 <= rows * cols <= 1 << 27:
            break
    case = {"op": op, "rows": rows, "cols": cols, "dtype": rng.choice(["f32", "f32", "bf16", "f16"])}
    if op == "reduce":
        case["axis"], case["kind"] = rng.choice([0, 1]), rng.choice(["sum", "max", "min"])
    if op == "copy":
        case["out"] = rng.choice([t for t in ("f32", "bf16", "f16", "fp8") if t != case["dtype"]]
                                 + [case["dtype"]])
        case["padded"] = rng.random() < 0.3
    return case


def draw(rng):
    kind = rng.random()
    return _draw_gemm(rng) if kind < 0.5 else _draw_attn(rng) if kind < 0.8 else _draw_tile(rng)


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _gen(seed, tag):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 16 + tag)
    return g


def _matrix(shape, dtype, gen, std):
    """Activations and weights N(0, std); f32 uniform in [-1, 1]; int8
    uniform in [-127, 127]; fp8 N(0, 1) scaled to amax 448 (with its factor)."""
    if dtype == "int8":
        return torch.randint(-127, 128, shape, generator=gen, device="cuda", dtype=torch.int8), 1.0
    if dtype == "f32":
        return torch.rand(shape, generator=gen, device="cuda") * 2 - 1, 1.0
    x = torch.randn(shape, generator=gen, device="cuda")
    if dtype == "fp8":
        scale = 448.0 / float(x.abs().max())
        return (x * scale).to(DTYPES["fp8"]), 1.0 / scale
    return (x * std).to(DTYPES[dtype]), 1.0


def _gemm_inputs(c, seed):
    ta, tb = c["layout"][0] == "t", c["layout"][1] == "t"
    m, n, k = c["m"], c["n"], c["k"]
    a, sa = _matrix((k, m) if ta else (m, k), c["dtype"], _gen(seed, 1), 1.0)
    b, sb = _matrix((n, k) if tb else (k, n), c["dtype"], _gen(seed, 2), 0.02)
    if not c["accumulate"]:
        out = torch.empty(m, n, dtype=DTYPES[c["out"]], device="cuda")
    elif c["out"] == "int32":
        out = torch.randint(-1000, 1000, (m, n), generator=_gen(seed, 3), device="cuda",
                            dtype=torch.int32)
    else:
        out = torch.randn(m, n, generator=_gen(seed, 3), device="cuda").to(DTYPES[c["out"]])
    return a, b, out, ta, tb, sa, sb


def _attn_inputs(c, seed):
    b, h, d, dt = c["batch"], c["heads"], c["head_dim"], DTYPES[c["dtype"]]

    def tensor(seq, tag):
        shape = (b, seq, h, d) if c["layout"] == "bshd" else (b, h, seq, d)
        x = torch.randn(shape, generator=_gen(seed, tag), device="cuda").to(dt)
        return x.transpose(1, 2) if c["layout"] == "bshd" else x

    q, k, v = tensor(c["seq_q"], 5), tensor(c["seq_k"], 6), tensor(c["seq_k"], 7)
    if c["k_transposed"]:
        k = k.transpose(-1, -2).contiguous()
    return q, k, v


def _tile_input(c, seed):
    g = _gen(seed, 11)
    cols = c["cols"] + (8 if c.get("padded") else 0)
    return torch.randn(c["rows"], cols, generator=g, device="cuda").to(DTYPES[c["dtype"]])[:, :c["cols"]]


def prepare(case, seed):
    c, op = dict(case), case["op"]
    if op == "gemm":
        a, b, out, ta, tb, sa, sb = _gemm_inputs(c, seed)
        s = {"op": op, "via": c["via"], "a": a, "b": b, "c": out, "ta": ta, "tb": tb, "sa": sa,
             "sb": sb, "clear": not c["accumulate"]}
        if c["via"] == "execute":  # the program, built once
            h = F.create_session()
            types = [h.memref_type(list(t.shape), IR_NAMES[n])
                     for t, n in ((a, c["dtype"]), (b, c["dtype"]), (out, c["out"]))]
            _, entry = h.new_kernel("gemm", types)
            h.create_gemm(*(entry.get_argument(i) for i in range(3)), trans_a=ta, trans_b=tb,
                          clear_accum=s["clear"])
            s["session"] = h
        return s
    if op == "attn":
        q, k, v = _attn_inputs(c, seed)
        o = torch.empty_strided(q.shape, q.stride(), dtype=DTYPES[c["out"]], device="cuda")
        lse = torch.empty(q.shape[:3], device="cuda") if c["lse"] else None
        return {"op": op, "q": q, "k": k, "v": v, "o": o, "lse": lse, "causal": c["causal"],
                "kt": c["k_transposed"]}
    if op == "fill":
        value = 0.25 * (1 + seed % 64)
        return {"op": op, "y": torch.empty(c["rows"], c["cols"], dtype=DTYPES[c["dtype"]],
                                           device="cuda"), "value": value}
    x = _tile_input(c, seed)
    if op == "reduce":
        out = torch.empty(c["rows"] if c["axis"] == 1 else c["cols"], dtype=x.dtype, device="cuda")
        return {"op": op, "x": x, "y": out, "kind": c["kind"], "axis": c["axis"]}
    return {"op": op, "x": x, "y": torch.empty(c["rows"], c["cols"], dtype=DTYPES[c["out"]],
                                               device="cuda")}


def run(s):
    op = s["op"]
    if op == "gemm":
        if s["via"] == "execute":
            return F.execute(s["session"].module, "gemm", [s["a"], s["b"], s["c"]],
                             scale_a=s["sa"], scale_b=s["sb"])
        return rt.gemm(s["a"], s["b"], s["c"], trans_a=s["ta"], trans_b=s["tb"],
                       clear_accum=s["clear"], scale_a=s["sa"], scale_b=s["sb"])
    if op == "attn":
        o = rt.attn_fwd(s["q"], s["k"], s["v"], s["o"], causal=s["causal"], lse=s["lse"],
                        k_transposed=s["kt"])
        return o if s["lse"] is None else (o, s["lse"])
    if op == "reduce":
        return rt.reduce(s["x"], s["y"], s["kind"], axis=s["axis"])
    if op == "copy":
        return rt.copy(s["x"], s["y"])
    return rt.fill(s["y"], s["value"])


# ---------------------------------------------------------------------------
# What a case takes, and what it gives
# ---------------------------------------------------------------------------
def _visible(c):
    """(query, key) pairs an attention case computes."""
    if not c["causal"]:
        return c["seq_q"] * c["seq_k"]
    first = c["seq_k"] - c["seq_q"] + 1  # keys the first query sees
    return c["seq_q"] * (first + c["seq_k"]) / 2


def work(case):
    c, op = case, case["op"]
    if op == "gemm":
        m, n, k, e, o = c["m"], c["n"], c["k"], BYTES[c["dtype"]], BYTES[c["out"]]
        return {"bytes": (m * k + n * k) * e + m * n * o * (2 if c["accumulate"] else 1),
                "flops": 2.0 * m * n * k}
    if op == "attn":
        bh, d, e = c["batch"] * c["heads"], c["head_dim"], BYTES[c["dtype"]]
        return {"bytes": bh * (c["seq_q"] * d * (e + BYTES[c["out"]]) + 2 * c["seq_k"] * d * e
                               + (4 * c["seq_q"] if c["lse"] else 0)),
                "flops": 4.0 * bh * d * _visible(c)}
    cells, e = c["rows"] * c["cols"], BYTES[c["dtype"]]
    if op == "reduce":
        return {"bytes": (cells + (c["rows"] if c["axis"] == 1 else c["cols"])) * e, "flops": cells}
    if op == "copy":
        return {"bytes": cells * (e + BYTES[c["out"]]), "flops": 0}
    return {"bytes": cells * e, "flops": 0}


def tolerance(case):
    """Tile ops follow one fixed order and rounding, and int8 products are
    whole numbers: exact.  The others allow about four times the largest error
    against 64 bits over 120 drawn cases: a GEMM's result is one rounding of
    an f32 sum (bf16 1.7e-3, f16 2.1e-4, f32 sums 1.6e-6 at the longest K);
    attention rounds the probabilities to the input type as well (bf16
    2.4e-3, f16 3.0e-4)."""
    c, op = case, case["op"]
    if op == "gemm":
        if c["out"] == "int32":
            return "exact"
        return {"rel": {"bf16": 7e-3, "f16": 9e-4, "f32": 7e-6}[c["out"]]}
    if op == "attn":
        return {"rel": {"bf16": 1e-2, "f16": 1.2e-3}[c["dtype"]]}
    return "exact"


def exact(case, seed):
    c, op = case, case["op"]
    if op == "gemm":
        if c["out"] == "int32":
            return None
        a, b, c0, ta, tb, sa, sb = _gemm_inputs(c, seed)
        x = (a.double().t() if ta else a.double()) @ (b.double().t() if tb else b.double())
        x *= sa * sb
        return x + c0.double() if c["accumulate"] else x
    if op == "attn":
        q, k, v = _attn_inputs(c, seed)
        sq, sk, scale = c["seq_q"], c["seq_k"], c["head_dim"] ** -0.5
        o = torch.empty(q.shape, dtype=torch.float64, device="cuda")
        lse = torch.empty(q.shape[:3], dtype=torch.float64, device="cuda")
        mask = None
        if c["causal"]:
            rows = torch.arange(sq, device="cuda")[:, None] + (sk - sq)
            mask = torch.arange(sk, device="cuda")[None, :] > rows
        for i in range(c["batch"]):
            for j in range(c["heads"]):
                kt = k[i, j].double() if c["k_transposed"] else k[i, j].double().t()
                s = (q[i, j].double() @ kt) * scale
                if mask is not None:
                    s.masked_fill_(mask, -math.inf)
                l = torch.logsumexp(s, dim=1)
                o[i, j] = torch.exp(s - l[:, None]) @ v[i, j].double()
                lse[i, j] = l
        return (o, lse) if c["lse"] else o
    if op == "fill":
        return torch.full((c["rows"], c["cols"]), 0.25 * (1 + seed % 64), dtype=torch.float64,
                          device="cuda")
    x = _tile_input(c, seed).double()
    if op == "copy":
        return x
    if c["kind"] == "sum":
        return x.sum(dim=c["axis"])
    return x.amax(dim=c["axis"]) if c["kind"] == "max" else x.amin(dim=c["axis"])
