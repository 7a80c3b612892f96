"""Performance cases of the HIP backend: what a program that uses it calls, over the sizes it calls it with.

Each case is one pass through the public ctypes binding (``dotcompute_amd.hip``) on inputs resident
on the GPU. ``listed()`` gives the fixed cases, ``draw()`` more of the same ranges, ``prepare()`` the
inputs of one case, ``run()`` one pass, ``exact()`` the same result in 64 bits from plain torch.

Kinds of cases:
  quickstart  VectorAdd, then Sum of its result (two dependent calls)
  sum         Sum over float32 (float64 accumulation) or int32 (exact, checked)
  to_array    Where -> Select -> ToArray, fused, order-preserving
  reduce      Where -> Select -> Sum with Count, then -> Max, over one source (two calls)
  gemm        row-major C = A B, float32, or bfloat16 inputs with a float32 result
  spmv        one y = A x from CSR arrays (float32, float64 or int32)
  plan        y = A x through a plan that was built once (float32)
  power       the 20-step normalised power iteration from CSR arrays
"""
import math

import numpy as np
import torch

from dotcompute_amd import hip

DEV = "cuda:0"
MAX_DEGREE = 4096  # SpMV graphs: out-degrees follow a Zipf law (alpha = 2) on [1, MAX_DEGREE]
ITERATIONS = 20

_E, _I, _S0 = hip.SRC_ELEM, hip.SRC_IMM, hip.SRC_S0
# Lambdas of the LINQ cases: (instructions, is the element type int32, share of the elements kept).
PROGRAMS = {
    # Where(x => x > 0f).Select(x => x * 2f + 1f)
    "affine": ([(hip.LOAD, _E, 0), (hip.CMP_GT, _I, 0.0), (hip.FILTER, _I, 0),
                (hip.LOAD, _E, 0), (hip.MUL, _I, 2.0), (hip.ADD, _I, 1.0), (hip.MAP, _I, 0)], False, 0.5),
    # Where(x => x > -0.5f && x < 0.5f).Select(x => x * x + x)
    "quadratic": ([(hip.LOAD, _E, 0), (hip.CMP_GT, _I, -0.5), (hip.CMP_LT, _I, 0.5, hip.CMP_AND), (hip.FILTER, _I, 0),
                   (hip.LOAD, _E, 0), (hip.MUL, _E, 0), (hip.ADD, _E, 0), (hip.MAP, _I, 0)], False, 0.5),
    # Where(x => x != 0f).Select(x => MathF.Sqrt(MathF.Abs(x)) / (x * x + 1f))
    "root": ([(hip.LOAD, _E, 0), (hip.CMP_NE, _I, 0.0), (hip.FILTER, _I, 0),
              (hip.LOAD, _E, 0), (hip.MUL, _E, 0), (hip.ADD, _I, 1.0), (hip.STORE_S0, _I, 0),
              (hip.LOAD, _E, 0), (hip.ABS, _I, 0), (hip.SQRT, _I, 0), (hip.DIV, _S0, 0), (hip.MAP, _I, 0)], False, 1.0),
    # Where(x => x % 2 == 0).Select(x => x * x)
    "evens": ([(hip.LOAD, _E, 0), (hip.REM, _I, 2), (hip.CMP_EQ, _I, 0), (hip.FILTER, _I, 0),
               (hip.LOAD, _E, 0), (hip.MUL, _E, 0), (hip.MAP, _I, 0)], True, 1001 / 2001),
    # Where(x => x > 0).Select(x => x * 3 - 1)
    "positive": ([(hip.LOAD, _E, 0), (hip.CMP_GT, _I, 0), (hip.FILTER, _I, 0),
                  (hip.LOAD, _E, 0), (hip.MUL, _I, 3), (hip.SUB, _I, 1), (hip.MAP, _I, 0)], True, 1000 / 2001),
}


def listed():
    return [
        # the README's first program: 100,000 floats added, then summed. Launches and latency.
        {"name": "quickstart_100k", "kind": "quickstart", "n": 100_000},
        # a checked Sum over an ordinary int column whose length is no multiple of anything
        {"name": "sum_i32_16m", "kind": "sum", "dtype": "i32", "n": 16_000_003, "offset": 0},
        # a filter-and-map over a small float column that starts inside a buffer (a slice)
        {"name": "array_affine_1m", "kind": "to_array", "program": "affine", "n": 1_000_003, "offset": 1},
        # the same over a column of 256M floats (1 GiB), the largest in use
        {"name": "array_affine_256m", "kind": "to_array", "program": "affine", "n": 1 << 28, "offset": 0},
        # a general float lambda: a range test and a polynomial, over a large ragged column
        {"name": "array_quadratic_60m", "kind": "to_array", "program": "quadratic", "n": 60_000_007, "offset": 0},
        # an int lambda with a remainder over a large column
        {"name": "array_evens_64m", "kind": "to_array", "program": "evens", "n": 1 << 26, "offset": 0},
        # two terminals over one mapped source (a column's total and its peak)
        {"name": "reduce_root_16m", "kind": "reduce", "program": "root", "n": 16_000_003, "offset": 0},
        # an ordinary float matrix product, every side odd
        {"name": "gemm_f32_odd", "kind": "gemm", "dtype": "f32", "m": 1_537, "n": 2_049, "k": 1_023},
        # the largest float product in use
        {"name": "gemm_f32_8192", "kind": "gemm", "dtype": "f32", "m": 8_192, "n": 8_192, "k": 8_192},
        # an ordinary bf16 product with sides that are multiples of 8 only
        {"name": "gemm_bf16_2000", "kind": "gemm", "dtype": "bf16", "m": 2_000, "n": 3_000, "k": 1_000},
        # one SpMV<double> over a graph of a million rows
        {"name": "spmv_f64_1m", "kind": "spmv", "dtype": "f64", "rows": 1_000_000},
        # PageRank-style power iteration over 16M rows (about 87M nonzeros), analysis included
        {"name": "power_16m", "kind": "power", "rows": 16_000_000},
    ]


def _log_size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["quickstart", "sum", "to_array", "to_array", "to_array", "reduce", "gemm", "gemm", "gemm", "spmv",
                       "plan", "power"])
    if kind == "quickstart":
        return {"kind": kind, "n": _log_size(rng, 100_000, 1 << 26)}
    if kind == "sum":
        return {"kind": kind, "dtype": rng.choice(["f32", "i32"]), "n": _log_size(rng, 300_000, 1 << 28),
                "offset": rng.choice([0, 0, 0, 1, 2, 3])}
    if kind in ("to_array", "reduce"):
        program = rng.choice(sorted(PROGRAMS))
        return {"kind": kind, "program": program, "n": _log_size(rng, 100_000, 1 << 28),
                "offset": rng.choice([0, 0, 0, 1, 2, 3])}
    if kind == "gemm":
        step = rng.choice([1, 1, 8, 64, 256])  # sides of real products: odd, or multiples of a tile
        while True:
            m, n, k = (max(step, _log_size(rng, 64, 8_192) // step * step) for _ in range(3))
            if m * n * k >= 1 << 20:
                return {"kind": kind, "dtype": rng.choice(["f32", "bf16"]), "m": m, "n": n, "k": k}
    if kind == "spmv":
        return {"kind": kind, "dtype": rng.choice(["f32", "f64", "i32"]), "rows": _log_size(rng, 20_000, 8_000_000)}
    return {"kind": kind, "rows": _log_size(rng, 50_000, 12_000_000)}


# ---- a program's state ---------------------------------------------------------------------------

_ctx = None


def context():
    """The program's one context, made on first use."""
    global _ctx
    if _ctx is None:
        _ctx = hip.Context(0)
    return _ctx


_DTYPES = {torch.float32: np.float32, torch.float64: np.float64, torch.int32: np.int32, torch.int64: np.int64,
           torch.bfloat16: np.uint16}


def _array(t):
    """The binding's view of a tensor's memory (the state keeps the tensor)."""
    dt = np.dtype(_DTYPES[t.dtype])
    return hip.DeviceArray(context(), t.data_ptr(), t.numel() * dt.itemsize, dt, tuple(t.shape))


class State:
    """Tensors, their views by the same name, and whatever else a pass needs."""

    def __init__(self, case):
        self.case, self.t, self.plan = case, {}, None

    def add(self, **tensors):
        for name, t in tensors.items():
            self.t[name] = t
            setattr(self, name, _array(t))

    def __del__(self):
        if self.plan is not None:
            self.plan.destroy()


def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _column(case, gen, dtype):
    """n elements starting `offset` elements into a buffer: U[-1, 1) floats, or ints in [-1000, 1000]."""
    n, off = case["n"], case.get("offset", 0)
    if dtype == "i32":
        base = torch.randint(-1000, 1001, (n + off,), device=DEV, dtype=torch.int32, generator=gen)
    else:
        base = torch.rand(n + off, device=DEV, generator=gen).mul_(2.0).sub_(1.0)
    return base[off:]


def _degree_cdf():
    w = torch.arange(1, MAX_DEGREE + 1, dtype=torch.float64).pow(-2.0)
    return torch.cumsum(w / w.sum(), 0)


def _mean_degree():
    w = [d ** -2.0 for d in range(1, MAX_DEGREE + 1)]
    return sum(d * x for d, x in zip(range(1, MAX_DEGREE + 1), w)) / sum(w)


def _graph(rows, gen, dtype):
    """A CSR graph: Zipf out-degrees, uniform columns without self-loops, values 1 / out-degree (or
    ints in [-1000, 1000])."""
    u = torch.rand(rows, device=DEV, dtype=torch.float64, generator=gen)
    deg = torch.searchsorted(_degree_cdf().to(DEV), u).clamp_(max=MAX_DEGREE - 1) + 1
    rp = torch.zeros(rows + 1, device=DEV, dtype=torch.int32)
    rp[1:] = torch.cumsum(deg, 0)
    row = torch.repeat_interleave(torch.arange(rows, device=DEV, dtype=torch.int32), deg)
    nnz = row.numel()
    col = torch.randint(0, rows - 1, (nnz,), device=DEV, dtype=torch.int32, generator=gen)
    col += (col >= row).to(torch.int32)
    if dtype == torch.int32:
        val = torch.randint(-1000, 1001, (nnz,), device=DEV, dtype=torch.int32, generator=gen)
    else:
        val = torch.repeat_interleave((1.0 / deg.to(torch.float64)).to(dtype), deg)
    return rp, col, val, row


def _inputs(case, seed):
    """The case's input tensors by name, from the seed alone."""
    gen, kind = _generator(seed), case["kind"]
    if kind == "quickstart":
        return {"a": _column(case, gen, "f32"), "b": _column(case, gen, "f32")}
    if kind == "sum":
        return {"x": _column(case, gen, case["dtype"])}
    if kind in ("to_array", "reduce"):
        return {"x": _column(case, gen, "i32" if PROGRAMS[case["program"]][1] else "f32")}
    if kind == "gemm":
        a = torch.randn(case["m"], case["k"], device=DEV, generator=gen)
        b = torch.randn(case["k"], case["n"], device=DEV, generator=gen)
        if case["dtype"] == "bf16":
            a, b = a.to(torch.bfloat16), b.to(torch.bfloat16)
        return {"a": a, "b": b}
    rows = case["rows"]
    dtype = {"f64": torch.float64, "i32": torch.int32}.get(case.get("dtype"), torch.float32)
    rp, col, val, row = _graph(rows, gen, dtype)
    if kind == "power":
        x = torch.full((rows,), 1.0 / rows, device=DEV)
    elif dtype == torch.int32:
        x = torch.randint(-1000, 1001, (rows,), device=DEV, dtype=dtype, generator=gen)
    else:
        x = torch.rand(rows, device=DEV, dtype=dtype, generator=gen)
    return {"rp": rp, "col": col, "val": val, "x": x, "row": row}


def _zeros(n, dtype):
    return torch.zeros(n, device=DEV, dtype=dtype)


def prepare(case, seed):
    ctx, kind = context(), case["kind"]
    inputs = _inputs(case, seed)
    inputs.pop("row", None)
    s = State(case)
    s.add(**inputs)
    if kind == "quickstart":
        s.add(r=_zeros(case["n"], torch.float32), total=_zeros(1, torch.float64))
    elif kind == "sum":
        s.add(total=_zeros(1, torch.int64 if case["dtype"] == "i32" else torch.float64), overflow=_zeros(1, torch.int32))
    elif kind in ("to_array", "reduce"):
        code, is_int, _ = PROGRAMS[case["program"]]
        s.chain = hip.LinqChain.assemble(code, int32=is_int)
        s.add(count=_zeros(1, torch.int64), count_max=_zeros(1, torch.int64))
        if kind == "to_array":  # a buffer for every element; what is past the kept ones stays zero
            s.add(out=_zeros(case["n"], torch.int32 if is_int else torch.float32))
        else:
            s.add(total=_zeros(1, torch.int64 if is_int else torch.float64), overflow=_zeros(1, torch.int32),
                  peak=_zeros(1, torch.int32 if is_int else torch.float32))
    elif kind == "gemm":
        s.add(c=_zeros(case["m"] * case["n"], torch.float32).view(case["m"], case["n"]))
    else:
        s.add(y=_zeros(case["rows"], s.t["val"].dtype))
        s.nnz = s.t["col"].numel()
        if kind == "power":
            s.add(v=_zeros(case["rows"], torch.float32), norm=_zeros(1, torch.float64))
        elif kind == "plan":
            torch.cuda.synchronize()  # the arrays are on torch's stream, the plan is built on the context's
            s.plan = ctx.spmv_plan(s.rp, s.col, s.val, case["rows"], case["rows"], s.nnz)
    torch.cuda.synchronize()
    return s


def run(s):
    ctx, case, t = context(), s.case, s.t
    kind = case["kind"]
    if kind == "quickstart":
        ctx.vector_add_f32(s.a, s.b, s.r)
        ctx.reduce_sum_f32(s.r, s.total)
        return t["r"], t["total"]
    if kind == "sum":
        if case["dtype"] == "i32":
            ctx.reduce_sum_i32(s.x, s.total, s.overflow)
            return t["total"], t["overflow"]
        ctx.reduce_sum_f32(s.x, s.total)
        return t["total"]
    if kind == "to_array":
        if PROGRAMS[case["program"]][1]:
            ctx.where_select_i32(s.chain, s.x, s.out, s.count, None)
        else:
            ctx.where_select_f32(s.chain, s.x, s.out, s.count)
        return t["out"], t["count"]
    if kind == "reduce":
        if PROGRAMS[case["program"]][1]:
            ctx.where_select_sum_i32(s.chain, s.x, s.total, s.count, s.overflow, None)
            ctx.where_select_minmax_i32(s.chain, s.x, hip.LINQ_MAX, s.peak, s.count_max, None)
            return t["total"], t["count"], t["peak"], t["count_max"], t["overflow"]
        ctx.where_select_sum_f32(s.chain, s.x, s.total, s.count)
        ctx.where_select_minmax_f32(s.chain, s.x, hip.LINQ_MAX, s.peak, s.count_max)
        return t["total"], t["count"], t["peak"], t["count_max"]
    if kind == "gemm":
        gemm = ctx.gemm_bf16 if case["dtype"] == "bf16" else ctx.gemm_f32
        gemm(s.a, s.b, s.c, case["m"], case["n"], case["k"])
        return t["c"]
    rows = case["rows"]
    if kind == "spmv":
        ctx.spmv_csr(s.rp, s.col, s.val, s.x, s.y, rows, rows, s.nnz)
        return t["y"]
    if kind == "plan":
        s.plan.execute(s.x, s.y)
        return t["y"]
    # the start vector is copied in on the context's stream, so a pass does not go on from the last one
    hip.check(hip.load().dc_hip_memcpy_d2d_async(ctx.handle, s.v.ptr, s.x.ptr, 4 * rows), "d2d copy")
    ctx.spmv_power_iterate_f32(s.rp, s.col, s.val, s.v, s.y, rows, s.nnz, ITERATIONS, s.norm)
    return t["v"], t["norm"]


def work(case):
    """Bytes and operations that no implementation can do without: each input read and each output
    written once (the power iteration: the matrix once per step)."""
    kind = case["kind"]
    if kind == "quickstart":
        return {"bytes": 12 * case["n"], "flops": 2 * case["n"]}
    if kind == "sum":
        return {"bytes": 4 * case["n"], "flops": case["n"]}
    if kind in ("to_array", "reduce"):
        kept = PROGRAMS[case["program"]][2] if kind == "to_array" else 0.0
        return {"bytes": 4 * case["n"] * (1.0 + kept), "flops": 2 * case["n"]}
    if kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": (2 if case["dtype"] == "bf16" else 4) * (m * k + k * n) + 4 * m * n, "flops": 2 * m * n * k}
    rows, nnz = case["rows"], case["rows"] * _mean_degree()
    size = 8 if case.get("dtype") == "f64" else 4
    once = nnz * (4 + size) + rows * (4 + 2 * size)
    times = ITERATIONS if kind == "power" else 1
    return {"bytes": times * once, "flops": times * 2 * nnz}


def tolerance(case):
    kind = case["kind"]
    if kind == "to_array" or (kind in ("sum", "spmv") and case["dtype"] == "i32"):
        return "exact"  # every float operation of a lambda rounds once; ints wrap
    if kind in ("quickstart", "sum", "reduce"):
        return {"rel": 1e-11}  # float64 totals of float32 values, in another order
    if kind == "spmv" and case["dtype"] == "f64":
        return {"rel": 1e-15, "max": 1e-13}  # long rows in another order
    if kind == "gemm":
        return {"rel": 1e-5, "max": 4e-4}  # float32 sums over up to 8,192 products
    return {"rel": 1e-6, "max": 4e-5}  # float32 sums over a row's products, long rows in another order


# ---- the same results in 64 bits -----------------------------------------------------------------


def _evaluate(program, x):
    """(kept elements, mapped, in float64) of a float column. The filter sees the float32 values."""
    if program == "affine":
        k = x[x > 0].double()
        return k * 2 + 1
    if program == "quadratic":
        k = x[(x > -0.5) & (x < 0.5)].double()
        return k * k + k
    k = x[x != 0].double()
    return k.abs().sqrt() / (k * k + 1)


def exact(case, seed):
    kind = case["kind"]
    inp = _inputs(case, seed)
    if kind == "quickstart":
        # the elements to be summed are the float32 results
        return inp["a"].double() + inp["b"].double(), (inp["a"] + inp["b"]).double().sum().reshape(1)
    if kind == "sum":
        return None if case["dtype"] == "i32" else inp["x"].double().sum().reshape(1)
    if kind in ("to_array", "reduce"):
        if PROGRAMS[case["program"]][1]:
            return None
        v = _evaluate(case["program"], inp["x"])
        if kind == "reduce":
            return v.sum().reshape(1), None, v.max().reshape(1), None
        out = torch.zeros(case["n"], device=DEV, dtype=torch.float64)
        out[:v.numel()] = v
        return out, None
    if kind == "gemm":
        return inp["a"].double() @ inp["b"].double()
    if case.get("dtype") == "i32":
        return None
    val, col, row = inp["val"].double(), inp["col"], inp["row"]

    def product(x):
        return torch.zeros_like(x).index_add_(0, row, val * x[col])

    x = inp["x"].double()
    if kind != "power":
        return product(x)
    for _ in range(ITERATIONS):
        y = product(x)
        norm = y.sum()
        x = y / norm
    return x, norm.reshape(1)
