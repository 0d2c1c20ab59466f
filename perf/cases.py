"""Performance cases of the library, each one call of a public entry point.

`listed()` gives the fixed cases, `draw(rng)` more of the same ranges; see the
comment at each.  Matrices are uniform on [-1, 1) (the tall case: normal, the
short operand scaled by 1/sqrt(k)), as in bench.py.
"""
import math

import torch

import sushiblas_amd as sbx

F32, F64 = "f32", "f64"


def _gemm(dtype, m, n, k, layout=0, ta=0, tb=0, alpha=1.0, beta=0.0, batch=1, relu=0,
          dist="uniform"):
    return {"op": "gemm", "dtype": dtype, "layout": layout, "ta": ta, "tb": tb, "m": m, "n": n,
            "k": k, "alpha": alpha, "beta": beta, "batch": batch, "relu": relu, "dist": dist}


def _gemv(dtype, m, n, layout=0, trans=0, alpha=1.0, beta=0.0):
    return {"op": "gemv", "dtype": dtype, "layout": layout, "ta": trans, "m": m, "n": n,
            "alpha": alpha, "beta": beta}


def _syrk(dtype, n, k, layout=0, upper=0, trans=0, alpha=1.0, beta=0.0):
    return {"op": "syrk", "dtype": dtype, "layout": layout, "upper": upper, "ta": trans, "n": n,
            "k": k, "alpha": alpha, "beta": beta}


def listed():
    return [
        # the smallest product of the benchmark: one call costs its latency
        {"name": "gemm_f32_512", **_gemm(F32, 512, 512, 512)},
        # a small ragged batch of rows through a weight stored n x k (a layer's forward call)
        {"name": "gemm_f32_37x1000x300", **_gemm(F32, 37, 1000, 300, tb=1)},
        # a dense layer with its ReLU in one call
        {"name": "gemm_relu_f32_512x1024x1024", **_gemm(F32, 512, 1024, 1024, relu=1)},
        # 24 independent layers of one shape (parallel inference), strided, with the ReLU
        {"name": "gemm_relu_f32_24x256x512x256", **_gemm(F32, 256, 512, 256, batch=24, relu=1)},
        # ragged sizes, leading dimensions without vector alignment, accumulating into C
        {"name": "gemm_f32_ragged", **_gemm(F32, 4095, 3001, 2047, ta=1, alpha=1.0, beta=1.0)},
        # the benchmark's headline
        {"name": "gemm_f32_8192", **_gemm(F32, 8192, 8192, 8192, alpha=1.5, beta=0.5)},
        # tall and skinny: a gigabyte of A against 64 columns
        {"name": "gemm_f32_tall", **_gemm(F32, 65536, 64, 4096, dist="tall")},
        # fp64, mid-size, ragged, column-major as a LAPACK-style caller stores it
        {"name": "gemm_f64_ragged", **_gemm(F64, 1500, 1300, 1023, layout=1, tb=1, beta=0.5)},
        # fp64 at the largest size
        {"name": "gemm_f64_8192", **_gemm(F64, 8192, 8192, 8192)},
        # matrix-vector products, one per direction and type: A is read once
        {"name": "gemv_f32_16384", **_gemv(F32, 16384, 16384)},
        {"name": "gemv_f64_t_16384x8192", **_gemv(F64, 16384, 8192, trans=1)},
        # Gram matrix, one triangle
        {"name": "syrk_f32_8192", **_syrk(F32, 8192, 8192)},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5)))))))


def draw(rng):
    """One more case: products of all transposes and both layouts from 64 to
    8192 on a side, strided batches of small ones, tall and wide ones with a
    short side of 8-64, GEMV from 64 to 16384 and SYRK from 64 to 8192; up to
    4e11 flop, as bench.py's list of problems for judging the kernel choice."""
    while True:
        kind = rng.choice(["gemm", "gemm", "gemm", "batch", "skinny", "gemv", "syrk"])
        dtype = F32 if rng.random() < 0.7 else F64
        layout, ta, tb, relu = (rng.randrange(2) for _ in range(4))
        alpha, beta = rng.choice([1.0, 1.5]), rng.choice([0.0, 0.5, 1.0])
        if kind == "gemm":
            c = _gemm(dtype, *(_log_int(rng, 64, 8192) for _ in range(3)), layout=layout, ta=ta,
                      tb=tb, alpha=alpha, beta=beta, relu=relu)
        elif kind == "batch":
            c = _gemm(dtype, *(_log_int(rng, 32, 1024) for _ in range(3)), layout=layout, ta=ta,
                      tb=tb, alpha=alpha, beta=beta, relu=relu,
                      batch=rng.choice([2, 3, 4, 7, 8, 16, 24, 32, 64]))
        elif kind == "skinny":
            long, short, k = _log_int(rng, 4096, 65536), _log_int(rng, 8, 64), _log_int(rng, 256, 4096)
            m, n = (long, short) if rng.random() < 0.5 else (short, long)
            c = _gemm(dtype, m, n, k, layout=layout, ta=ta, tb=tb, alpha=alpha, beta=beta, dist="tall")
        elif kind == "gemv":
            c = _gemv(dtype, _log_int(rng, 64, 16384), _log_int(rng, 64, 16384), layout=layout,
                      trans=ta, alpha=alpha, beta=beta)
        else:
            c = _syrk(dtype, _log_int(rng, 64, 8192), _log_int(rng, 64, 8192), layout=layout,
                      upper=relu, trans=ta, alpha=alpha, beta=beta)
        w = work(c)
        if w["flops"] <= 4e11 and w["bytes"] <= 1.2e9:
            return c


def _esize(case):
    return 4 if case["dtype"] == F32 else 8


def _tdt(case):
    return torch.float32 if case["dtype"] == F32 else torch.float64


def _code(case):
    return sbx.F32 if case["dtype"] == F32 else sbx.F64


def _stored(case, trans, rows, cols):
    """Row-major view dimensions of an operand's storage (column-major storage
    of r x c is row-major storage of c x r) and so its leading dimension."""
    r, c = (cols, rows) if trans else (rows, cols)
    return (r, c) if case["layout"] == 0 else (c, r)


def work(case):
    e, op = _esize(case), case["op"]
    reads_c = 1 if case["beta"] != 0 else 0
    if op == "gemm":
        m, n, k, b = case["m"], case["n"], case["k"], case["batch"]
        return {"bytes": b * (m * k + k * n + m * n * (1 + reads_c)) * e, "flops": 2.0 * m * n * k * b}
    if op == "gemv":
        m, n = case["m"], case["n"]
        x, y = (m, n) if case["ta"] else (n, m)
        return {"bytes": (m * n + x + y * (1 + reads_c)) * e, "flops": 2.0 * m * n}
    n, k = case["n"], case["k"]
    return {"bytes": (n * k + n * (n + 1) // 2 * (1 + reads_c)) * e, "flops": float(n) * (n + 1) * k}


def prepare(case, seed):
    """The operands as device buffers, and the call's arguments."""
    gen = torch.Generator(device="cuda").manual_seed(int(seed))

    def make(shape, normal=0.0):
        t = torch.empty(shape, dtype=_tdt(case), device="cuda")
        return t.normal_(0.0, normal, generator=gen) if normal else t.uniform_(-1.0, 1.0, generator=gen)

    s = {"case": case}
    if case["op"] == "gemm":
        m, n, k, b = case["m"], case["n"], case["k"], case["batch"]
        tall = case["dist"] == "tall"
        # the long operand is N(0, 1), the short one N(0, 1/k)
        na, nb = (0.0, 0.0) if not tall else (1.0, k ** -0.5) if m >= n else (k ** -0.5, 1.0)
        s["A"] = make((b,) + _stored(case, case["ta"], m, k), na)
        s["B"] = make((b,) + _stored(case, case["tb"], k, n), nb)
        s["C"] = make((b,) + _stored(case, 0, m, n))
    elif case["op"] == "gemv":
        m, n = case["m"], case["n"]
        x, y = (m, n) if case["ta"] else (n, m)
        s["A"] = make((1,) + _stored(case, 0, m, n))
        s["B"], s["C"] = make((x,)), make((y,))
    else:
        n, k = case["n"], case["k"]
        s["A"] = make((1,) + _stored(case, case["ta"], n, k))
        s["C"] = make((1, n, n))
    return s


def run(state):
    c, A, C = state["case"], state["A"], state["C"]
    if c["op"] == "gemv":
        sbx.gemv(_code(c), c["layout"], c["ta"], c["m"], c["n"], c["alpha"], A, A.shape[2],
                 state["B"], 1, c["beta"], C, 1)
        return C
    if c["op"] == "syrk":
        sbx.syrk(_code(c), c["layout"], c["upper"], c["ta"], c["n"], c["k"], c["alpha"], A,
                 A.shape[2], 0, c["beta"], C, c["n"], 0)
        return C
    B, batch = state["B"], c["batch"]
    args = (_code(c), c["layout"], c["ta"], c["tb"], c["m"], c["n"], c["k"], c["alpha"], A,
            A.shape[2], A.shape[1] * A.shape[2] if batch > 1 else 0, B, B.shape[2],
            B.shape[1] * B.shape[2] if batch > 1 else 0, c["beta"], C, C.shape[2],
            C.shape[1] * C.shape[2] if batch > 1 else 0, batch)
    if c["relu"]:
        sbx.gemm_fused(*args)
    else:
        sbx.gemm_ex(*args)
    return C


def exact(case, seed):
    s = prepare(case, seed)
    A, C = s["A"].double(), s["C"].double()
    col = case["layout"] == 1
    if case["op"] == "gemv":
        a = A[0].t() if col else A[0]
        y = (a.t() if case["ta"] else a) @ s["B"].double()
        return case["alpha"] * y + (case["beta"] * C if case["beta"] else 0.0)

    def logical(x, trans):
        x = x.transpose(1, 2) if col else x
        return x.transpose(1, 2) if trans else x

    if case["op"] == "syrk":
        a = logical(A, case["ta"])[0]
        full = case["alpha"] * (a @ a.t()) + (case["beta"] * logical(C, 0)[0] if case["beta"] else 0.0)
        i = torch.arange(case["n"], device="cuda")
        keep = (i[None, :] >= i[:, None]) if case["upper"] else (i[None, :] <= i[:, None])
        out = torch.where(keep, full, logical(C, 0)[0])
        return (out.t() if col else out).contiguous()[None]
    B = s["B"].double()
    out = torch.empty(case["batch"], case["m"], case["n"], dtype=torch.float64, device="cuda")
    for z in range(case["batch"]):
        out[z] = case["alpha"] * (logical(A, case["ta"])[z] @ logical(B, case["tb"])[z])
    if case["beta"]:
        out += case["beta"] * logical(C, 0)
    if case["relu"]:
        out = out.clamp_min(0.0)
    return (out.transpose(1, 2) if col else out).contiguous()


def tolerance(case):
    """A sum of k products in order, in fp32, is off by 1.8e-8 sqrt(k) of its
    norm (measured: 8.1e-7 at k = 2047, 1.15e-6 at 4096, 1.6e-6 at 8192); four
    times that, and not below what the rounding of a few terms gives.  fp64
    scales with its unit roundoff, 2^-29 of fp32's."""
    depth = case["k"] if case["op"] != "gemv" else (case["m"] if case["ta"] else case["n"])
    rel = max(7.2e-8 * math.sqrt(depth), 6e-7)
    return {"rel": rel if case["dtype"] == F32 else rel * 2.0 ** -29}
