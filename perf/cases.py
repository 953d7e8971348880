"""The workloads this framework's speed is judged by, each one call of a public
entry point of sile_amd on operands that are resident on the GPU.

The listed cases are the benchmark's own configurations (GEMM, causal
attention and row softmax at 8192, the DSL matmul at 512), the shapes a
serving program has between them (a few rows against a large weight matrix,
short sequences, row widths that are no multiple of anything) and the two DSL
programs with a kernel of their own (the online-softmax attention, the mlp
example's matvec).  draw() gives further cases of the same families.

`work` counts each operand read once and each result written once, and the
arithmetic of the definition (causal attention: the pairs below the diagonal).
"""
from __future__ import annotations

import math

import torch

from sile_amd import _abi as hip

DEV = "cuda"
TYPES = {"f32": (hip.F32, torch.float32), "f16": (hip.F16, torch.float16),
         "bf16": (hip.BF16, torch.bfloat16), "fp8": (hip.F8E4M3, torch.float8_e4m3fn)}
SIZE = {"f32": 4, "f16": 2, "bf16": 2, "fp8": 1}


def listed():
    return [
        # the headline GEMM: a large dense layer, weights stored [N, K]
        {"name": "gemm_bf16_8192", "op": "gemm", "dtype": "bf16", "out": "bf16", "layout": "col",
         "m": 8192, "n": 8192, "k": 8192},
        # the same layer quantised per tensor to e4m3
        {"name": "gemm_fp8_8192", "op": "gemm", "dtype": "fp8", "out": "bf16", "layout": "col",
         "m": 8192, "n": 8192, "k": 8192},
        # an ordinary layer in the canonical matmul's own layout ([K, N]) at
        # sizes no tile divides (a batch of 1333 rows)
        {"name": "gemm_f16_brow_1333", "op": "gemm", "dtype": "f16", "out": "f16", "layout": "row",
         "m": 1333, "n": 3000, "k": 2056},
        # decoding: a few rows against a whole weight matrix
        {"name": "gemm_bf16_decode_16", "op": "gemm", "dtype": "bf16", "out": "bf16",
         "layout": "col", "m": 16, "n": 8192, "k": 8192},
        # the DSL matmul program, 32 x 32 tiles, bit for bit the CPU backend's
        {"name": "dsl_matmul_f32_512", "op": "dsl_matmul", "m": 512, "n": 512, "k": 512,
         "tile": 32, "bk": 32},
        # long-context prefill: the headline attention
        {"name": "attn_f16_causal_8192", "op": "attn", "dtype": "f16", "b": 4, "h": 32,
         "s": 8192, "d": 128, "causal": True},
        # short-sequence encoding: odd length, full attention, narrow heads
        {"name": "attn_bf16_1000_d64", "op": "attn", "dtype": "bf16", "b": 2, "h": 8,
         "s": 1000, "d": 64, "causal": False},
        # the DSL attention program (fp32, K transposed), one head
        {"name": "attn_f32_dsl_1024x4096", "op": "attn_f32", "nq": 1024, "nk": 4096, "d": 128},
        # the headline row softmax
        {"name": "softmax_f16_8192", "op": "softmax", "dtype": "f16", "out": "f16",
         "rows": 8192, "cols": 8192, "pad": 0},
        # a contiguous score matrix whose width is odd
        {"name": "softmax_f32_4097x3001", "op": "softmax", "dtype": "f32", "out": "f32",
         "rows": 4097, "cols": 3001, "pad": 0},
        # row statistics of a 16-bit activation matrix
        {"name": "reduce_sum_bf16_16384x1000", "op": "reduce", "dtype": "bf16", "how": "sum",
         "rows": 16384, "cols": 1000, "pad": 0},
        # the smallest call: the mlp example's matvec
        {"name": "matvec_f32_1024", "op": "matvec", "m": 1024, "k": 1024, "bk": 8},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _extent(rng, lo, hi, unit):
    """A size spread over the logarithm of [lo, hi]: half of them multiples of
    `unit`, the others whatever comes."""
    x = _log(rng, lo, hi)
    if rng.random() < 0.5:
        x = max(lo, x // unit * unit)
    return x


def draw(rng):
    op = rng.choice(["gemm", "gemm", "gemm_few_rows", "dsl_matmul", "attn", "attn", "attn_f32",
                     "softmax", "softmax", "reduce", "matvec"])
    if op in ("gemm", "gemm_few_rows"):
        dtype = rng.choice(["bf16", "f16", "fp8"])
        few = op == "gemm_few_rows"
        return {"op": "gemm", "dtype": dtype,
                "out": rng.choice([dtype if dtype != "fp8" else "bf16"] * 3 + ["f32"]),
                "layout": "col" if few or dtype == "fp8" or rng.random() < 0.6 else "row",
                "m": _extent(rng, 1, 128, 8) if few else _extent(rng, 128, 8192, 64),
                "n": _extent(rng, 512, 16384, 128) // 8 * 8 if few else _extent(rng, 128, 8192, 64),
                "k": _extent(rng, 512, 16384, 128) if few else _extent(rng, 128, 8192, 64)}
    if op == "dsl_matmul":
        tile, bk = rng.choice([16, 32, 64]), rng.choice([8, 16, 32])
        m, n = (max(1, _log(rng, 64, 2048) // tile) * tile for _ in range(2))
        return {"op": "dsl_matmul", "m": m, "n": n, "k": _extent(rng, 64, 2048, 32), "tile": tile,
                "bk": bk}
    if op == "attn":
        s = _extent(rng, 64, 8192, 64)
        d, causal = rng.choice([32, 40, 64, 64, 72, 80, 96, 128, 128, 128]), rng.random() < 0.6
        most = (1 << 40) // (s * s * d) // (1 if causal else 2)  # the listed 128 heads of 8192 x 128
        heads = min(rng.choice([2, 5, 8, 12, 16, 24, 32, 64, 128]), most)
        b = rng.choice([x for x in (1, 2, 4) if heads % x == 0])
        return {"op": "attn", "dtype": rng.choice(["f16", "bf16"]), "b": b, "h": heads // b,
                "s": s, "d": d, "causal": causal}
    if op == "attn_f32":
        return {"op": "attn_f32", "nq": _extent(rng, 64, 4096, 64),
                "nk": _extent(rng, 64, 8192, 64), "d": rng.choice([32, 64, 80, 100, 128])}
    if op in ("softmax", "reduce"):
        cols = _extent(rng, 32, 65536, 64)
        rows = min(_log(rng, 64, 16384), (1 << 26) // cols)
        case = {"op": op, "rows": rows, "cols": cols, "pad": rng.choice([0, 0, 0, 8, 5])}
        if op == "softmax":
            case["dtype"], case["out"] = rng.choice([("f16", "f16"), ("bf16", "bf16"),
                                                     ("f32", "f32"), ("f16", "f32")])
        else:
            case["dtype"], case["how"] = rng.choice(["f32", "f16", "bf16"]), rng.choice(["max", "sum"])
        return case
    return {"op": "matvec", "m": _extent(rng, 512, 8192, 64), "k": _extent(rng, 512, 8192, 64),
            "bk": rng.choice([4, 8, 16, 32, 64])}


def _normal(gen, shape, sigma=1.0):
    return torch.randn(shape, generator=gen, device=DEV, dtype=torch.float32) * sigma


def _pitched(rows, ld, cols, dtype, gen, sigma):
    """A [rows, cols] matrix of N(0, sigma^2) in rows of `ld` elements."""
    t = torch.zeros((rows, ld), device=DEV, dtype=dtype)
    t[:, :cols] = _normal(gen, (rows, cols), sigma).to(dtype)
    return t


def _round_up(x, unit):
    return (x + unit - 1) // unit * unit


def _quantised(x):
    """Per-tensor e4m3: codes and the scale amax / 448."""
    scale = float(x.abs().max()) / 448.0
    return (x / scale).to(torch.float8_e4m3fn), scale


def prepare(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    if not torch.cuda.is_initialized():
        torch.cuda.init()
    hip.init(torch.cuda.current_device())
    st = dict(case)
    op = case["op"]
    if op == "gemm":
        m, n, k, dt = case["m"], case["n"], case["k"], TYPES[case["dtype"]][1]
        # operand rows start on 16-byte boundaries, as the entry point asks
        ld = _round_up(k, 16 // SIZE[case["dtype"]])
        row_major_b = case["layout"] == "row"
        st["sa"] = st["sb"] = 1.0
        if case["dtype"] == "fp8":
            (qa, st["sa"]), (qb, st["sb"]) = (_quantised(_normal(gen, (r, k))) for r in (m, n))
            st["a"] = torch.zeros((m, ld), device=DEV, dtype=torch.uint8)
            st["b"] = torch.zeros((n, ld), device=DEV, dtype=torch.uint8)
            st["a"][:, :k] = qa.view(torch.uint8)
            st["b"][:, :k] = qb.view(torch.uint8)
        else:
            st["a"] = _pitched(m, ld, k, dt, gen, k ** -0.5)
            if row_major_b:
                st["b"] = _pitched(k, n, n, dt, gen, k ** -0.5)
            else:
                st["b"] = _pitched(n, ld, k, dt, gen, k ** -0.5)
        st["lda"], st["ldb"] = ld, n if row_major_b else ld
        st["c"] = torch.zeros((m, n), device=DEV, dtype=TYPES[case["out"]][1])
    elif op == "dsl_matmul":
        m, n, k = case["m"], case["n"], case["k"]
        st["a"], st["b"] = (torch.rand(s, generator=gen, device=DEV) * 2 - 1 for s in ((m, k), (k, n)))
        st["c"] = torch.zeros((m, n), device=DEV)
    elif op == "attn":
        shape = (case["b"], case["h"], case["s"], case["d"])
        st["q"], st["k"], st["v"] = (_normal(gen, shape).to(TYPES[case["dtype"]][1]) for _ in range(3))
        st["o"] = torch.zeros_like(st["q"])
    elif op == "attn_f32":
        nq, nk, d = case["nq"], case["nk"], case["d"]
        st["q"], st["kt"], st["v"] = (_normal(gen, s) for s in ((nq, d), (d, nk), (nk, d)))
        st["o"] = torch.zeros((nq, d), device=DEV)
    elif op in ("softmax", "reduce"):
        rows, cols, ld = case["rows"], case["cols"], case["cols"] + case["pad"]
        st["x"] = _pitched(rows, ld, cols, TYPES[case["dtype"]][1], gen, 2.0)
        st["y"] = (torch.zeros((rows, cols), device=DEV, dtype=TYPES[case["out"]][1])
                   if op == "softmax" else torch.zeros(rows, device=DEV))
    else:
        st["x"], st["y"] = _normal(gen, (case["m"], case["k"])), _normal(gen, (case["k"],))
        st["out"] = torch.zeros(case["m"], device=DEV)
    return st


def run(st):
    op = st["op"]
    if op == "gemm":
        t = TYPES[st["dtype"]][0]
        hip.gemm(t, t, TYPES[st["out"]][0], st["m"], st["n"], st["k"], st["a"].data_ptr(),
                 st["lda"], hip.ROW_MAJOR, st["b"].data_ptr(), st["ldb"],
                 hip.ROW_MAJOR if st["layout"] == "row" else hip.COL_MAJOR, st["c"].data_ptr(),
                 st["n"], st["sa"], st["sb"])
        return st["c"]
    if op == "dsl_matmul":
        m, n, k, tile = st["m"], st["n"], st["k"], st["tile"]
        hip.kernel_matmul([st["a"].data_ptr(), st["b"].data_ptr(), st["c"].data_ptr()],
                          (m // tile) * (n // tile), [m, k, k, n, m, n], tile, tile, st["bk"])
        return st["c"]
    if op == "attn":
        hip.flash_attn_fwd(TYPES[st["dtype"]][0], st["b"], st["h"], st["s"], st["d"],
                           st["q"].data_ptr(), st["k"].data_ptr(), st["v"].data_ptr(),
                           st["o"].data_ptr(), st["d"] ** -0.5, st["causal"])
        return st["o"]
    if op == "attn_f32":
        nq, nk, d = st["nq"], st["nk"], st["d"]
        hip.attention_f32_kt(nq, nk, d, st["q"].data_ptr(), d, st["kt"].data_ptr(), nk,
                             st["v"].data_ptr(), d, st["o"].data_ptr(), d, d ** -0.5, -1e30)
        return st["o"]
    if op == "softmax":
        ld = st["cols"] + st["pad"]
        hip.softmax_rows(TYPES[st["dtype"]][0], TYPES[st["out"]][0], st["rows"], st["cols"],
                         st["x"].data_ptr(), ld, st["y"].data_ptr(), st["cols"])
        return st["y"]
    if op == "reduce":
        hip.reduce_rows(hip.REDUCE_SUM if st["how"] == "sum" else hip.REDUCE_MAX,
                        TYPES[st["dtype"]][0], st["rows"], st["cols"], st["x"].data_ptr(),
                        st["cols"] + st["pad"], st["y"].data_ptr())
        return st["y"]
    hip.matvec_f32(st["m"], st["k"], st["bk"], st["x"].data_ptr(), st["k"], st["y"].data_ptr(),
                   st["out"].data_ptr())
    return st["out"]


def work(case):
    op = case["op"]
    if op == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": SIZE[case["dtype"]] * (m + n) * k + SIZE[case["out"]] * m * n,
                "flops": 2 * m * n * k}
    if op == "dsl_matmul":
        m, n, k = case["m"], case["n"], case["k"] // case["bk"] * case["bk"]
        return {"bytes": 4 * ((m + n) * k + m * n), "flops": 2 * m * n * k}
    if op == "attn":
        heads, s, d = case["b"] * case["h"], case["s"], case["d"]
        pairs = s * (s + 1) // 2 if case["causal"] else s * s
        return {"bytes": 4 * 2 * heads * s * d, "flops": 4 * d * heads * pairs}
    if op == "attn_f32":
        nq, nk, d = case["nq"], case["nk"], case["d"]
        return {"bytes": 4 * d * (2 * nq + 2 * nk), "flops": 4 * d * nq * nk}
    if op == "softmax":
        rows, cols = case["rows"], case["cols"]
        return {"bytes": rows * cols * (SIZE[case["dtype"]] + SIZE[case["out"]]),
                "flops": 5 * rows * cols}
    if op == "reduce":
        rows, cols = case["rows"], case["cols"]
        return {"bytes": rows * cols * SIZE[case["dtype"]] + 4 * rows, "flops": rows * cols}
    m, k = case["m"], case["k"] // case["bk"] * case["bk"]
    return {"bytes": 4 * (m * k + k + m), "flops": 2 * m * k}


def tolerance(case):
    """About four times what the path measures against 64 bits: the rounding
    of a 16-bit result (and of attention's 16-bit probabilities), a few ulp of
    a 32-bit one (more where thousands of terms are summed; the fp8 matrix
    instruction aligns its products before it adds them, 1.5e-5).  The DSL
    matmul, the matvec and the row max are defined bit for bit."""
    op = case["op"]
    if op in ("dsl_matmul", "matvec") or (op == "reduce" and case["how"] == "max"):
        return "exact"
    out = case["out"] if op in ("gemm", "softmax") else case["dtype"] if op == "attn" else "f32"
    if out == "bf16":
        return {"rel": 8e-3}
    if out == "f16":
        return {"rel": 1e-3}
    if op == "gemm":
        return {"rel": 6e-5 if case["dtype"] == "fp8" else 2e-6}
    return {"rel": 6e-6 if op == "attn_f32" else 1e-6}


def _dense(t, cols):
    return t[:, :cols].double()


def exact(case, seed):
    st = prepare(case, seed)
    op = case["op"]
    if op == "gemm":
        k = case["k"]
        if case["dtype"] == "fp8":
            a, b = (_dense(st[x].view(torch.float8_e4m3fn).float(), k) for x in ("a", "b"))
            return (a @ b.t().contiguous()) * (st["sa"] * st["sb"])
        b = st["b"].double() if case["layout"] == "row" else _dense(st["b"], k).t().contiguous()
        return _dense(st["a"], k) @ b
    if op == "dsl_matmul":
        k = case["k"] // case["bk"] * case["bk"]
        return st["a"][:, :k].double() @ st["b"][:k].double()
    if op == "attn":
        s, d = case["s"], case["d"]
        q, k, v = (st[x].reshape(-1, s, d) for x in ("q", "k", "v"))
        out = torch.empty(q.shape, device=DEV, dtype=torch.float64)
        above = torch.ones((s, s), device=DEV, dtype=torch.bool).triu(1) if case["causal"] else None
        for i in range(q.shape[0]):
            p = q[i].double() @ k[i].double().t().contiguous() * d ** -0.5
            if above is not None:
                p.masked_fill_(above, -math.inf)
            out[i] = torch.softmax(p, 1) @ v[i].double()
        return out.reshape(st["q"].shape)
    if op == "attn_f32":
        p = st["q"].double() @ st["kt"].double() * case["d"] ** -0.5
        return torch.softmax(p, 1) @ st["v"].double()
    if op == "softmax":
        return torch.softmax(_dense(st["x"], case["cols"]), 1)
    if op == "reduce":
        x = _dense(st["x"], case["cols"])
        return x.sum(1) if case["how"] == "sum" else x.amax(1)
    k = case["k"] // case["bk"] * case["bk"]
    return st["x"][:, :k].double() @ st["y"][:k].double()
