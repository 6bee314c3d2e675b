"""The calls a program makes into this library, as cases to time: GEMM (16-bit, 8-bit, float32), GEMM with a fused
bias and activation, block-scaled GEMM, GEMV and the DLRM dot interaction as a training step makes it (forward, then
backward).  The listed cases stand for the ranges below; draw() gives further cases of the same ranges.

  kind      ranges
  gemm      F16 / BF16 (results in F32 or the operands' type), I8 -> I32, E4M3 / E5M2 -> F32, F32; A and B row- or
            column-major; m, n, k of 256 to 8192 in steps of 16 (32 along k for the 8-bit types), F32 up to 2048; few
            token rows (16 to 128) against a weight matrix of up to 14336 x 8192; alpha = beta = 1 or 2, or no C
  bias_act  F16 / BF16, GELU or ReLU and a bias, 16 to 4096 token rows, weights of 1024 to 14336 by 1024 to 8192
  mx        E4M3 / E5M2 with block scales, 16 to 4096 token rows, the same weights
  gemv      F16, 1, 2, 4 or 8 right-hand sides, 1024 to 16384 rows, k of 1024 to 16384 in steps of 8
  dlrm      F16 / F32, 8 to 128 features of 16 to 256 elements, batches of 512 to 65536; 129 to 1024 features of up to
            1024 elements, batches of 16 to 64
"""
import math

import torch

import rocwmma_amd as rw

IN = {"f16": rw.F16, "bf16": rw.BF16, "e4m3": rw.E4M3, "e5m2": rw.E5M2, "i8": rw.I8, "f32": rw.F32, "i32": rw.I32}
TORCH = {"f16": torch.float16, "bf16": torch.bfloat16, "e4m3": torch.float8_e4m3fn, "e5m2": torch.float8_e5m2, "i8": torch.int8,
         "f32": torch.float32, "i32": torch.int32}
SIZE = {"f16": 2, "bf16": 2, "e4m3": 1, "e5m2": 1, "i8": 1, "f32": 4, "i32": 4}
LAYOUT = {"row": rw.ROW_MAJOR, "col": rw.COL_MAJOR}
ACT = {"gelu": rw.ACT_GELU, "relu": rw.ACT_RELU}


def _gemm(dtype, out, a, b, m, n, k, alpha=1.0, beta=0.0):
    return {"kind": "gemm", "dtype": dtype, "out": out, "a": a, "b": b, "m": m, "n": n, "k": k, "alpha": alpha, "beta": beta}


def _bias_act(dtype, out, act, m, n, k):
    return {"kind": "bias_act", "dtype": dtype, "out": out, "act": act, "m": m, "n": n, "k": k}


def _mx(dtype, m, n, k):
    return {"kind": "mx", "dtype": dtype, "m": m, "n": n, "k": k}


def _gemv(m, k, ncols):
    return {"kind": "gemv", "m": m, "k": k, "ncols": ncols}


def _dlrm(dtype, m, k, batch):
    return {"kind": "dlrm", "dtype": dtype, "m": m, "k": k, "batch": batch}


def listed():
    cases = [
        # the smallest call: one 256^3 product with C, as the reference's first sample makes it; launch latency
        ("gemm_f16_256", _gemm("f16", "f32", "row", "col", 256, 256, 256, 2.0, 2.0)),
        # the largest: the benchmark's 8192^3, one of its layout pairs
        ("gemm_bf16_8192", _gemm("bf16", "f32", "row", "row", 8192, 8192, 8192, 1.0, 1.0)),
        # a layer whose sizes fill no tile and whose K ends inside a stage
        ("gemm_bf16_ragged", _gemm("bf16", "bf16", "row", "col", 2000, 3056, 1360)),
        # single precision, as the reference's blocked sgemm sample
        ("gemm_f32_2048", _gemm("f32", "f32", "row", "col", 2048, 2048, 2048, 2.0, 2.0)),
        # decode: sixteen token rows against a quantised MLP weight
        ("gemm_i8_m16", _gemm("i8", "i32", "row", "col", 16, 14336, 4096)),
        # a chunk of a prompt through an MLP layer with bias and activation
        ("bias_gelu_f16_m512", _bias_act("f16", "f16", "gelu", 512, 14336, 4096)),
        # batched decode in block-scaled fp8, scales as they come
        ("mx_e4m3_m128", _mx("e4m3", 128, 14336, 4096)),
        # a few right-hand sides against a f16 weight
        ("gemv_n4", _gemv(14336, 4096, 4)),
        # recommendation model, training step at the benchmark's batch
        ("dlrm_f16_b2048", _dlrm("f16", 27, 128, 2048)),
        # the same in single precision, a batch larger than the caches
        ("dlrm_f32_b65536", _dlrm("f32", 27, 128, 65536)),
        # feature count and embedding width that are no power of two
        ("dlrm_f16_odd", _dlrm("f16", 41, 72, 8192)),
        # the reference's largest DLRM test size
        ("dlrm_f16_m1024", _dlrm("f16", 1024, 1024, 64)),
    ]
    return [dict(c, name=name) for name, c in cases]


def _log(rng, low, high, step):
    """A multiple of `step` in low..high, spread evenly over the logarithm."""
    v = math.exp(rng.uniform(math.log(low), math.log(high)))
    return max(low, min(high, int(v) // step * step))


def _rows(rng):
    return _log(rng, 16, 4096, 16)


def draw(rng):
    what = rng.choice(["gemm", "gemm", "gemm", "few_rows", "f32", "bias_act", "mx", "gemv", "dlrm", "dlrm", "dlrm_large"])
    a, b = rng.choice(["row", "col"]), rng.choice(["row", "col"])
    if what == "gemm":
        dtype, out = rng.choice([("f16", "f32"), ("f16", "f16"), ("bf16", "f32"), ("bf16", "bf16"), ("i8", "i32"), ("e4m3", "f32"), ("e5m2", "f32")])
        # at most a quarter of the largest listed product: sizes off the tiles are far slower than it
        while True:
            m, n = _log(rng, 256, 8192, 16), _log(rng, 256, 8192, 16)
            k = _log(rng, 256, 8192, 16 if SIZE[dtype] == 2 else 32)
            if m * n * k <= 1 << 35:
                break
        alpha, beta = rng.choice([(1.0, 0.0), (1.0, 1.0), (2.0, 2.0)])
        return _gemm(dtype, out, a, b, m, n, k, alpha, beta)
    if what == "few_rows":
        dtype, out = rng.choice([("i8", "i32"), ("e4m3", "f32"), ("f16", "f32"), ("bf16", "f32")])
        return _gemm(dtype, out, "row", "col", 16 * rng.randint(1, 8), _log(rng, 1024, 14336, 16), _log(rng, 1024, 8192, 128))
    if what == "f32":
        return _gemm("f32", "f32", a, b, _log(rng, 256, 2048, 16), _log(rng, 256, 2048, 16), _log(rng, 256, 2048, 16), 2.0, rng.choice([0.0, 2.0]))
    if what == "bias_act":
        dtype, out = rng.choice([("f16", "f16"), ("bf16", "bf16"), ("bf16", "f32")])
        return _bias_act(dtype, out, rng.choice(["gelu", "relu"]), _rows(rng), _log(rng, 1024, 14336, 16), _log(rng, 1024, 8192, 32))
    if what == "mx":
        return _mx(rng.choice(["e4m3", "e5m2"]), _rows(rng), _log(rng, 1024, 14336, 16), _log(rng, 1024, 8192, 128))
    if what == "gemv":
        return _gemv(_log(rng, 1024, 16384, 1), _log(rng, 1024, 16384, 8), rng.choice([1, 2, 4, 8]))
    dtype = rng.choice(["f16", "f32"])
    if what == "dlrm":
        m, k = _log(rng, 8, 128, 1), rng.choice([16, 32, 64, 64, 128, 128, 256, 8 * rng.randint(2, 32)])
        # at most the elements of the largest listed batch
        most = max(512, min(65536, 27 * 128 * 65536 // (max(m, 16) * (max(k, 32) + m))))
        return _dlrm(dtype, m, k, _log(rng, 512, most, 1))
    m, k = _log(rng, 129, 1024, 1), _log(rng, 64, 1024, 8)
    return _dlrm(dtype, m, k, _log(rng, 16, 64, 1))


def _values(gen, dtype, shape, scale):
    if dtype == "i8":
        return torch.randint(-127, 128, shape, generator=gen, device="cuda", dtype=torch.int8)
    return torch.empty(shape, device="cuda").normal_(0.0, scale, generator=gen).to(TORCH[dtype])


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    s = dict(case)
    kind = case["kind"]
    if kind == "gemm":
        m, n, k, dtype, out = case["m"], case["n"], case["k"], case["dtype"], case["out"]
        s["A"] = _values(gen, dtype, (m, k) if case["a"] == "row" else (k, m), 1.0)
        s["B"] = _values(gen, dtype, (k, n) if case["b"] == "row" else (n, k), 1.0 if SIZE[dtype] == 1 else 1.0 / math.sqrt(k))
        s["C"] = None
        if case["beta"] != 0.0:
            s["C"] = (torch.randint(-1000, 1001, (m, n), generator=gen, device="cuda", dtype=torch.int32) if out == "i32"
                      else _values(gen, out, (m, n), 1.0))
        s["D"] = torch.empty((m, n), dtype=TORCH[out], device="cuda")
    elif kind == "bias_act":
        m, n, k = case["m"], case["n"], case["k"]
        s["A"] = _values(gen, case["dtype"], (m, k), 1.0)
        s["B"] = _values(gen, case["dtype"], (n, k), 1.0 / math.sqrt(k))
        s["bias"] = _values(gen, "f32", (n,), 0.5)
        s["D"] = torch.empty((m, n), dtype=TORCH[case["out"]], device="cuda")
    elif kind == "mx":
        m, n, k = case["m"], case["n"], case["k"]
        s["A"] = _values(gen, case["dtype"], (m, k), 1.0)
        s["B"] = _values(gen, case["dtype"], (n, k), 1.0)
        s["scale_a"] = torch.randint(123, 128, (m, k // 32), generator=gen, device="cuda", dtype=torch.uint8)
        s["scale_b"] = torch.randint(118, 123, (n, k // 32), generator=gen, device="cuda", dtype=torch.uint8)
        s["D"] = torch.empty((m, n), device="cuda")
        s["workspace"] = torch.empty(rw.gemm_mx_workspace_size(m, n, k), dtype=torch.uint8, device="cuda")
    elif kind == "gemv":
        s["A"] = _values(gen, "f16", (case["m"], case["k"]), 1.0 / math.sqrt(case["k"]))
        s["X"] = _values(gen, "f16", (case["ncols"], case["k"]), 1.0)
        s["Y"] = torch.zeros((case["ncols"], case["m"]), device="cuda")
    else:
        m, k, batch, dtype = case["m"], case["k"], case["batch"], case["dtype"]
        width = k + m * (m - 1) // 2
        s["features"] = _values(gen, dtype, (batch, m, k), k ** -0.25)
        s["upstream"] = _values(gen, dtype, (batch, width), 1.0 / math.sqrt(m))
        s["out"] = torch.empty((batch, width), dtype=TORCH[dtype], device="cuda")
        s["grad"] = torch.empty((batch, m, k), dtype=TORCH[dtype], device="cuda")
        s["mlp_grad"] = torch.empty((batch, k), dtype=TORCH[dtype], device="cuda")
    return s


def run(s):
    kind = s["kind"]
    if kind == "gemm":
        return rw.gemm(IN[s["dtype"]], IN[s["out"]], LAYOUT[s["a"]], LAYOUT[s["b"]], rw.ROW_MAJOR, s["m"], s["n"], s["k"],
                       s["A"], s["B"], s["C"], s["D"], s["alpha"], s["beta"])
    if kind == "bias_act":
        return rw.gemm_bias_act(IN[s["dtype"]], IN[s["out"]], rw.ROW_MAJOR, rw.COL_MAJOR, rw.ROW_MAJOR, s["m"], s["n"], s["k"],
                                s["A"], s["B"], None, s["D"], 1.0, 0.0, s["bias"], ACT[s["act"]])
    if kind == "mx":
        return rw.gemm_mx(IN[s["dtype"]], rw.ROW_MAJOR, rw.COL_MAJOR, rw.ROW_MAJOR, s["m"], s["n"], s["k"], s["A"], s["scale_a"],
                          s["B"], s["scale_b"], None, s["D"], 1.0, 0.0, s["workspace"])
    if kind == "gemv":
        return rw.gemv(s["m"], s["k"], s["ncols"], s["A"], s["X"], s["Y"])
    dtype = IN[s["dtype"]]
    rw.dlrm_fwd(s["features"], s["out"], s["m"], s["k"], s["batch"], dtype)
    rw.dlrm_bwd(s["features"], s["upstream"], s["grad"], s["mlp_grad"], s["m"], s["k"], s["batch"], dtype)
    return {"out": s["out"], "grad": s["grad"], "mlp_grad": s["mlp_grad"]}


def work(case):
    kind = case["kind"]
    if kind == "gemv":
        m, k, c = case["m"], case["k"], case["ncols"]
        return {"bytes": 2 * m * k + 2 * k * c + 4 * m * c, "flops": 2 * m * k * c}
    if kind == "dlrm":
        m, k, batch, size = case["m"], case["k"], case["batch"], SIZE[case["dtype"]]
        width = k + m * (m - 1) // 2
        # forward: features in, row out; backward: features and upstream row in, gradient and bottom-MLP gradient out
        # (Z is symmetric: half of its products; the gradient takes all of G)
        return {"bytes": batch * size * (3 * m * k + 2 * width + k), "flops": batch * k * m * (m - 1 + 2 * (m - 1))}
    m, n, k = case["m"], case["n"], case["k"]
    size = SIZE[case["dtype"]]
    byts = (m * k + k * n) * size
    if kind == "mx":
        byts += (m + n) * (k // 32) + 4 * m * n
    elif kind == "bias_act":
        byts += 4 * n + m * n * SIZE[case["out"]]
    else:
        byts += m * n * SIZE[case["out"]] * (2 if case["beta"] != 0.0 else 1)
    return {"bytes": byts, "flops": 2 * m * n * k}


def tolerance(case):
    """About four times the relative error measured against the same product in float64 (listed and drawn cases): 5.7e-7
    for float32 results, 1.3e-5 where the matrix cores add fp8 products (they align the products of an instruction to
    the largest one), 2.1e-4 / 1.7e-3 for results rounded to f16 / bf16."""
    out = case.get("out", case["dtype"] if case["kind"] == "dlrm" else "f32")
    if out == "i32":
        return "exact"
    if case.get("dtype") in ("e4m3", "e5m2"):
        return {"rel": 5e-5}
    return {"rel": {"f32": 3e-6, "f16": 8e-4, "bf16": 6.6e-3}[out]}
