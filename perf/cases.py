"""The work a user of this package has it do, as cases that can be timed and compared: GEMM of every operand type, 2:4 sparse
GEMM, the DLRM dot interaction in both directions and the matrix-vector product, from calls of a few microseconds to 8192^3.

`listed()` names the cases, `draw()` gives further ones of the same ranges, `prepare()` makes what a program holds before the
call (operands, outputs, the workspace it keeps for its shape), `run()` is one call through the public entry points.
"""
import numpy as np
import torch

import rocwmma_amd as R

DTYPES = {"f16": R.F16, "bf16": R.BF16, "e4m3": R.E4M3, "i8": R.I8, "f32": R.F32, "i32": R.I32, "f64": R.F64}
TORCH = {"f16": torch.float16, "bf16": torch.bfloat16, "e4m3": torch.float8_e4m3fn, "i8": torch.int8, "f32": torch.float32,
         "i32": torch.int32, "f64": torch.float64}
BYTES = {"f16": 2, "bf16": 2, "e4m3": 1, "i8": 1, "f32": 4, "i32": 4, "f64": 8}
LAYOUT = {"row": R.ROW_MAJOR, "col": R.COL_MAJOR}


def _gemm(name, dtype, out, m, n, k, a="row", b="col", alpha=1.0, beta=0.0):
    return {"name": name, "op": "gemm", "dtype": dtype, "out": out, "m": m, "n": n, "k": k, "a": a, "b": b,
            "alpha": alpha, "beta": beta}


def _sparse(name, dtype, out, m, n, k, b="col"):
    return {"name": name, "op": "sparse", "dtype": dtype, "out": out, "m": m, "n": n, "k": k, "b": b}


def _dlrm(name, op, dtype, m, k, batch):
    return {"name": name, "op": op, "dtype": dtype, "m": m, "k": k, "batch": batch}


def _gemv(name, dtype, m, k, a):
    return {"name": name, "op": "gemv", "dtype": dtype, "m": m, "k": k, "a": a}


def listed():
    return [
        # the smallest call: one 256^3 product with both scalars and C, where latency and host time are what counts
        _gemm("gemm_f16_256", "f16", "f32", 256, 256, 256, alpha=2.0, beta=2.0),
        # the largest: the benchmark's own 8192^3, A col-major, B row-major
        _gemm("gemm_f16_8192", "f16", "f16", 8192, 8192, 8192, a="col", b="row"),
        # a layer of a network in training: ragged against every tile edge and every K stage, gradients in bf16
        _gemm("gemm_bf16_ragged", "bf16", "bf16", 2832, 4624, 3080, a="row", b="row"),
        # quantized inference, a size of the reference's benchmark list
        _gemm("gemm_i8_5120", "i8", "i32", 5120, 5120, 5120),
        # decoding: a batch of 64 rows against an fp8 weight matrix, K split over the workspace that the program keeps
        _gemm("gemm_e4m3_decode", "e4m3", "f32", 64, 8192, 8192),
        # single precision at an ordinary size of the reference's benchmark list
        _gemm("gemm_f32_2560", "f32", "f32", 2560, 2560, 2560),
        # 2:4 structured sparsity at the benchmark's size
        _sparse("sparse_i8_4096", "i8", "i32", 4096, 4096, 8192),
        # recommendation: the benchmark's dot interaction at the training batch
        _dlrm("dlrm_fwd_f16", "dlrm_fwd", "f16", 27, 128, 65536),
        # its gradient for a ragged batch of fewer and narrower features, in single precision
        _dlrm("dlrm_bwd_f32_ragged", "dlrm_bwd", "f32", 21, 64, 20011),
        # many features: the sizes of the reference's own tests beside 32 x 128, both directions
        _dlrm("dlrm_fwd_f16_wide", "dlrm_fwd", "f16", 1024, 1024, 64),
        _dlrm("dlrm_bwd_bf16_wide", "dlrm_bwd", "bf16", 320, 192, 96),
        # matrix times vector, a ragged matrix in the sample's orientation
        _gemv("gemv_f32_ragged", "f32", 6152, 11012, "col"),
    ]


def _log(rng, lo, hi, step):
    """A multiple of `step` in [lo, hi], evenly spread over the logarithm."""
    v = int(round(lo * (hi / lo) ** rng.random() / step)) * step
    return min(hi, max(lo, v))


def draw(rng):
    family = rng.choice(["gemm", "gemm", "gemm", "gemm", "small", "decode", "sparse", "dlrm", "dlrm", "wide", "wide", "gemv", "gemv"])
    layouts = [("row", "col"), ("col", "row"), ("row", "row"), ("col", "col")]
    if family in ("gemm", "small"):
        dtype, out = rng.choice([("f16", "f16"), ("f16", "f32"), ("bf16", "bf16"), ("bf16", "f32"), ("i8", "i32"), ("e4m3", "f32"),
                                 ("f32", "f32"), ("f64", "f64")])
        hi = {"f32": 3584, "f64": 2816}.get(dtype, 8192) if family == "gemm" else 768
        lo = 512 if family == "gemm" else 64
        m, n, k = (_log(rng, lo, hi, 16) for _ in range(3))
        a, b = rng.choice(layouts)
        alpha, beta = rng.choice([(1.0, 0.0), (1.0, 0.0), (1.0, 0.0), (2.0, 2.0)])
        case = _gemm("", dtype, out, m, n, k, a, b, alpha, beta)
    elif family == "decode":
        dtype, out = rng.choice([("f16", "f16"), ("bf16", "bf16"), ("i8", "i32"), ("e4m3", "f32")])
        a, b = rng.choice(layouts)
        case = _gemm("", dtype, out, _log(rng, 16, 256, 16), _log(rng, 1024, 16384, 16), _log(rng, 1024, 16384, 16), a, b)
    elif family == "sparse":
        dtype, out = rng.choice([("i8", "i32"), ("e4m3", "f32"), ("f16", "f32"), ("bf16", "f32")])
        case = _sparse("", dtype, out, _log(rng, 256, 6144, 16), _log(rng, 256, 6144, 16), _log(rng, 512, 8192, 128),
                       rng.choice(["col", "row"]))
    elif family == "dlrm":
        case = _dlrm("", rng.choice(["dlrm_fwd", "dlrm_bwd"]), rng.choice(["f16", "bf16", "f32"]), rng.randint(4, 32),
                     rng.choice([32, 64, 128]), _log(rng, 512, 65536, 1))
    elif family == "wide":
        m, k = _log(rng, 48, 1024, 16), _log(rng, 64, 1024, 16)
        most = max(4, min(1024, (64 << 20) // (m * k), (16 << 20) // (m * m)))
        case = _dlrm("", rng.choice(["dlrm_fwd", "dlrm_bwd"]), rng.choice(["f16", "bf16", "f32"]), m, k, _log(rng, 4, most, 1))
    else:
        dtype = rng.choice(["f32", "f32", "f64"])
        case = _gemv("", dtype, _log(rng, 256, 16384, 4), _log(rng, 256, 16384, 4), rng.choice(["row", "col"]))
    del case["name"]
    return case


def _operand(shape, dtype, gen):
    """What the path meets in earnest: weights and activations around zero, quantized values over their whole range."""
    if dtype == "i8":
        return torch.randint(-128, 128, shape, dtype=torch.int8, device="cuda", generator=gen)
    if dtype == "e4m3":
        return torch.randn(shape, device="cuda", generator=gen).clamp_(-448.0, 448.0).to(torch.float8_e4m3fn)
    wide = torch.float64 if dtype == "f64" else torch.float32
    return torch.rand(shape, dtype=wide, device="cuda", generator=gen).mul_(2.0).sub_(1.0).to(TORCH[dtype])


def _output(shape, dtype):
    return torch.zeros(shape, dtype=TORCH[dtype], device="cuda")


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    op, dtype = case["op"], case["dtype"]
    if op in ("gemm", "sparse"):
        m, n, k, out = case["m"], case["n"], case["k"], case["out"]
        b = _operand((k * n,), dtype, gen)
        d = _output((m, n), out)
        if op == "sparse":
            # a pruned weight matrix: of every four neighbours along K two stay, at any positions; compressed once on the host
            dense = _operand((m, k // 4, 4), dtype, gen)
            keep = torch.rand((m, k // 4, 4), device="cuda", generator=gen).argsort(dim=2) < 2
            bits = dense.view(torch.int8 if BYTES[dtype] == 1 else torch.int16) * keep
            host = np.ascontiguousarray(bits.reshape(m, k).cpu().numpy()).view(np.uint8 if BYTES[dtype] == 1 else np.uint16)
            values, meta = R.compress_24(host)
            a = torch.from_numpy(values.view(np.int8 if BYTES[dtype] == 1 else np.int16)).cuda()
            return {"call": "gemm", "d": d, "args": (DTYPES[dtype], DTYPES[out], m, n, k, a, b, None, d, 1.0, 0.0),
                    "kw": {"layout_a": R.ROW_MAJOR, "layout_b": LAYOUT[case["b"]], "a_meta": torch.from_numpy(meta).cuda()}}
        a = _operand((m * k,), dtype, gen)
        c = None
        if case["beta"] != 0.0:
            c = torch.randint(-1000, 1000, (m, n), dtype=torch.int32, device="cuda", generator=gen) if out == "i32" else _operand((m, n), out, gen)
        args = (DTYPES[dtype], DTYPES[out], m, n, k, a, b, c, d, case["alpha"], case["beta"])
        kw = {"layout_a": LAYOUT[case["a"]], "layout_b": LAYOUT[case["b"]]}
        # the workspace a program keeps beside the weights, of the size that the library asks for
        plan = R.gemm_query(R.gemm_args(*args, layout_c=R.ROW_MAJOR, layout_d=R.ROW_MAJOR, workspace_bytes=2**64 - 1, **kw))
        if plan.workspace_bytes:
            kw["workspace"] = torch.empty(plan.workspace_bytes, dtype=torch.uint8, device="cuda")
        return {"call": "gemm", "d": d, "args": args, "kw": kw}
    if op == "gemv":
        m, k = case["m"], case["k"]
        a, x = _operand((m * k,), dtype, gen), _operand((k,), dtype, gen)
        y = _output(m, dtype)
        kw = {}
        need = R.gemv_workspace_bytes(LAYOUT[case["a"]], m, k, BYTES[dtype])
        if need:
            kw["workspace"] = torch.empty(need, dtype=torch.uint8, device="cuda")
        return {"call": "dgemv" if dtype == "f64" else "gemv", "d": y, "args": (LAYOUT[case["a"]], m, k, a, x, None, y), "kw": kw}
    m, k, batch = case["m"], case["k"], case["batch"]
    width = k + m * (m - 1) // 2
    x = torch.randn((batch, m, k), device="cuda", generator=gen).to(TORCH[dtype])
    if op == "dlrm_fwd":
        out = _output((batch, width), dtype)
        return {"call": "dlrm_fwd", "d": out, "args": (DTYPES[dtype], x, out, m, k, batch), "kw": {}}
    up = torch.randn((batch, width), device="cuda", generator=gen).to(TORCH[dtype])
    mlp, grad = _output((batch, k), dtype), _output((batch, m, k), dtype)
    return {"call": "dlrm_bwd", "d": (mlp, grad), "args": (DTYPES[dtype], x, up, mlp, grad, m, k, batch), "kw": {}}


def run(state):
    getattr(R, state["call"])(*state["args"], **state["kw"])
    return state["d"]


def work(case):
    op, s = case["op"], BYTES[case["dtype"]]
    if op in ("gemm", "sparse"):
        m, n, k, so = case["m"], case["n"], case["k"], BYTES[case["out"]]
        if op == "sparse":  # kept values and their index bits; the multiplications that are left
            return {"bytes": m * k // 2 * s + m * k // 8 + k * n * s + m * n * so, "flops": m * n * k}
        return {"bytes": (m * k + k * n) * s + m * n * so * (2 if case["beta"] != 0.0 else 1), "flops": 2 * m * n * k}
    if op == "gemv":
        return {"bytes": (case["m"] * case["k"] + case["m"] + case["k"]) * s, "flops": 2 * case["m"] * case["k"]}
    m, k, batch = case["m"], case["k"], case["batch"]
    width = k + m * (m - 1) // 2
    if op == "dlrm_fwd":
        return {"bytes": batch * (m * k + width) * s, "flops": batch * m * (m - 1) * k}
    return {"bytes": batch * (2 * m * k + width + k) * s, "flops": 2 * batch * m * (m - 1) * k}


def tolerance(case):
    """About four times what the present kernels differ from a 64-bit evaluation of the same inputs: the rounding of the
    result for 16-bit results, the order of the sums for 32- and 64-bit ones, and for e4m3 operands the sums inside the matrix
    core, which keep less than 32 bits."""
    out = case.get("out", case["dtype"])
    if out == "i32":
        return "exact"
    if case["dtype"] == "e4m3":
        return {"rel": 6e-5, "max": 8e-4}
    return {"f16": {"rel": 8e-4, "max": 2e-3}, "bf16": {"rel": 7e-3, "max": 1.6e-2}, "f32": {"rel": 5e-6, "max": 4e-5},
            "f64": {"rel": 5e-15, "max": 4e-14}}[out]
