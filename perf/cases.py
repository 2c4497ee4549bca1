"""The work that users of this library have it do, as cases that can be timed and compared.

Every case is one call (or one solver run) through the C ABI of include/mpres_hip.h, by way of
the ctypes binding mpres-blas_amd/mpres.py. Device memory belongs to the caller: mp_array_t and
mp_float_t buffers are torch tensors whose addresses the calls take. Values are u * 2^e with u
uniform in [-1, 1) and an integer exponent e uniform in a range, as in the benchmark and tests.
Calls whose results leave multiple precision (reductions, products, the solver) end with the
export to doubles that such a program does (mp_get_d); axpy and SpMV are steps inside other
computations and keep their results in place.

Outputs are the results in full: residues, signs, exponents, interval evaluations, and the
exported doubles. exact() gives the doubles; the other fields depend on the residue number
system's own rounding order and have no value outside it.
"""
import ctypes as C
import importlib.util
import math
import os

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _load():
    spec = importlib.util.spec_from_file_location("mpres", os.path.join(ROOT, "mpres-blas_amd", "mpres.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


mp = _load()
SETS = {106: "8_2double", 212: "16_4double", 424: "32_8double"}
MODULI = {106: 8, 212: 16, 424: 32}
DEV = "cuda"
_contexts = {}


def context(bits):
    """One context per precision, kept for the life of the program, as a user's program does."""
    if bits not in _contexts:
        _contexts[bits] = mp.Context(SETS[bits])
    return _contexts[bits]


# ---------------------------------------------------------------- cases
def listed():
    return [
        # the smallest calls: a short vector's dot, where launches and the serial trees count
        {"name": "dot_106_1k", "op": "dot", "bits": 106, "n": 1003, "grid": 256, "block": 64, "inc": 1, "e": 20},
        # the benchmark's dot
        {"name": "dot_106_64k", "op": "dot", "bits": 106, "n": 65536, "grid": 256, "block": 64, "inc": 1, "e": 20},
        # the benchmark's long dot
        {"name": "dot_106_16m", "op": "dot", "bits": 106, "n": 1 << 24, "grid": 256, "block": 64, "inc": 1, "e": 20},
        # vector update on a strided (row of a matrix) x of odd length
        {"name": "axpy_212_1m", "op": "axpy", "bits": 212, "n": 1000003, "incx": 2, "incy": 1, "e": 20},
        # the benchmark's gemv at its full size
        {"name": "gemv_424_4096", "op": "gemv", "bits": 424, "trans": False, "m": 4096, "n": 4096, "block": 32, "e": 30},
        # A^T x of a tall ragged matrix (normal equations, least squares)
        {"name": "gemv_t_106_1500", "op": "gemv", "bits": 106, "trans": True, "m": 1501, "n": 777, "block": 32, "e": 20},
        # the benchmark's gemm
        {"name": "gemm_424_512", "op": "gemm", "bits": 424, "m": 512, "n": 512, "k": 512, "e": 30},
        # the reference tests' 300 x 300 product, not a multiple of any tile, at the recommended precision
        {"name": "gemm_212_300", "op": "gemm", "bits": 212, "m": 300, "n": 300, "k": 300, "e": 20},
        # the benchmark's SpMV: 10^6 rows of power-law lengths, 8 threads per row
        {"name": "spmv_212_1m", "op": "spmv", "bits": 212, "rows": 1000000, "tpr": 8, "e": 10},
        # a whole solve: preconditioned CG on a 2D grid, 20 iterations
        {"name": "pcg_212_20k", "op": "cg", "bits": 212, "grid": 141, "iters": 20},
        # the benchmark's exact-sum gemm (precision form)
        {"name": "mfma_106_2048", "op": "mfma", "bits": 106, "m": 2048, "n": 2048, "k": 2048, "ta": False, "tb": False,
         "e": 8},
        # a batch of many small uneven dots and gemvs, one plan and one launch
        {"name": "batch_212_1024", "op": "batch", "bits": 212, "count": 1024, "e": 20},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["dot", "dot", "axpy", "gemv", "gemv", "gemm", "gemm", "spmv", "cg", "mfma", "batch"])
    bits = rng.choice([106, 212, 424])
    if op == "dot":
        grid, block = rng.choice([(256, 64), (64, 64), (128, 128), (32, 256), (512, 32)])
        return {"op": op, "bits": bits, "n": _log(rng, 100, {106: 1 << 24, 212: 1 << 21, 424: 1 << 21}[bits]),
                "grid": grid, "block": block, "inc": rng.choice([1, 1, 2]), "e": rng.choice([8, 20, 60])}
    if op == "axpy":
        return {"op": op, "bits": bits, "n": _log(rng, 100, {106: 1 << 24, 212: 1 << 23, 424: 1 << 22}[bits]),
                "incx": rng.choice([1, 2]), "incy": rng.choice([1, 3]), "e": rng.choice([8, 20, 60])}
    if op == "gemv":
        top = {106: 2048, 212: 1536, 424: 4096}[bits]
        return {"op": op, "bits": bits, "trans": rng.choice([False, True]), "m": _log(rng, 32, top),
                "n": _log(rng, 32, top), "block": rng.choice([8, 32, 64]), "e": rng.choice([8, 20, 30])}
    if op == "gemm":
        top = {106: 320, 212: 320, 424: 512}[bits]
        return {"op": op, "bits": bits, "m": _log(rng, 16, top), "n": _log(rng, 16, top), "k": _log(rng, 16, top),
                "e": rng.choice([8, 20, 30])}
    if op == "spmv":
        return {"op": op, "bits": bits, "rows": _log(rng, 1000, 100000 if bits == 106 else 1000000),
                "tpr": rng.choice([1, 4, 8, 16]), "e": rng.choice([10, 20])}
    if op == "cg":
        return {"op": op, "bits": bits, "grid": _log(rng, 30, 160),
                "iters": rng.randint(*{106: (8, 20), 212: (8, 16), 424: (2, 4)}[bits])}
    if op == "mfma":
        return {"op": op, "bits": rng.choice([106, 424]), "m": _log(rng, 64, 2048), "n": _log(rng, 64, 2048),
                "k": _log(rng, 64, 2048), "ta": rng.choice([False, True]), "tb": rng.choice([False, True]),
                "e": rng.choice([8, 60])}
    return {"op": "batch", "bits": 212, "count": _log(rng, 64, 1024), "e": rng.choice([8, 20])}


# ---------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def values(g, count, e):
    """count doubles u * 2^k, u uniform in [-1, 1), k uniform in [-e, e]"""
    u = torch.rand(count, generator=g, device=DEV, dtype=torch.float64) * 2 - 1
    k = torch.randint(-e, e + 1, (count,), generator=g, device=DEV, dtype=torch.int32)
    return torch.ldexp(u, k)


class Array:
    """An mp_array_t of `size` numbers in torch memory, filled from doubles (or with zeros)."""

    def __init__(self, bits, size, x=None):
        n = MODULI[bits]
        self.bits, self.size = bits, size
        self.digits = torch.zeros((size, n), dtype=torch.int32, device=DEV)
        self.sign = torch.zeros(size, dtype=torch.int32, device=DEV)
        self.exp = torch.zeros(size, dtype=torch.int32, device=DEV)
        self.eval = torch.zeros((2 * size, 2), dtype=torch.int64, device=DEV)  # {double frac; long exp}
        self.buf = torch.empty((size, 4), dtype=torch.int32, device=DEV)
        self.len = torch.tensor([size], dtype=torch.int32, device=DEV)
        self.c = self.view(0)
        if x is not None:
            c = context(bits)
            mp.check(c.L.mpres_array_set_d(c.h, C.byref(self.c), x.data_ptr(), size, None))

    def view(self, at):
        """the mp_array_t that starts at element `at` (its upper bounds stay `len` behind its lower ones)"""
        n = self.digits.shape[1]
        return mp.MpArray(self.digits.data_ptr() + 4 * n * at, self.sign.data_ptr() + 4 * at,
                          self.exp.data_ptr() + 4 * at, self.eval.data_ptr() + 16 * at, self.buf.data_ptr() + 16 * at,
                          self.len.data_ptr())

    @property
    def ref(self):
        return C.byref(self.c)

    def fields(self):
        return {"digits": self.digits, "sign": self.sign, "exp": self.exp,
                "eval_frac": self.eval.view(torch.float64)[:, 0], "eval_exp": self.eval[:, 1]}


class Records:
    """`size` mp_float_t records in torch memory, filled from doubles (or zero)."""

    def __init__(self, bits, size, x=None):
        self.n = MODULI[bits]
        self.mem = torch.zeros((size, 4 * self.n + 40), dtype=torch.uint8, device=DEV)
        self.ptr = self.mem.data_ptr()
        if x is not None:
            c = context(bits)
            mp.check(c.L.mpres_set_d(c.h, self.ptr, x.data_ptr(), size, None))

    def fields(self):
        n, i, q = self.n, self.mem.view(torch.int32), self.mem.view(torch.int64)
        f = self.mem.view(torch.float64)
        at = n // 2 + 1
        return {"digits": i[:, :n], "sign": i[:, n], "exp": i[:, n + 1], "low_frac": f[:, at], "low_exp": q[:, at + 1],
                "up_frac": f[:, at + 2], "up_exp": q[:, at + 3]}


def powerlaw(g, rows, kmax=1024, alpha=1.6138):
    """CSR matrix: row lengths of P(k) ~ k^-alpha on [1, kmax] (mean 16), uniform columns ascending in the row"""
    p = torch.arange(1, kmax + 1, device=DEV, dtype=torch.float64) ** -alpha
    cdf = torch.cumsum(p / p.sum(), 0)
    k = torch.searchsorted(cdf, torch.rand(rows, generator=g, device=DEV, dtype=torch.float64)).clamp(max=kmax - 1) + 1
    irp = torch.zeros(rows + 1, dtype=torch.int64, device=DEV)
    irp[1:] = torch.cumsum(k, 0)
    nnz = int(irp[-1])
    row = torch.repeat_interleave(torch.arange(rows, device=DEV), k)
    col = torch.randint(0, rows, (nnz,), generator=g, device=DEV)
    col = torch.sort(row * rows + col).values - row * rows
    vals = torch.rand(nnz, generator=g, device=DEV, dtype=torch.float64) * 2 - 1
    return irp.to(torch.int32), col.to(torch.int32), vals


def grid_laplacian(g):
    """5-point stencil on a g x g grid, shifted by one: CSR on the device"""
    i = torch.arange(g * g, device=DEV)
    x, y = i % g, i // g
    cols = torch.stack([i - g, i - 1, i, i + 1, i + g], 1)
    live = torch.stack([y > 0, x > 0, x >= 0, x < g - 1, y < g - 1], 1)
    vals = torch.tensor([-1.0, -1.0, 5.0, -1.0, -1.0], dtype=torch.float64, device=DEV).expand(g * g, 5)
    irp = torch.zeros(g * g + 1, dtype=torch.int32, device=DEV)
    irp[1:] = torch.cumsum(live.sum(1), 0)
    return irp, cols[live].to(torch.int32), vals[live].contiguous()


def batch_sizes(case):
    """problem i even: a dot's length, log-uniform in [64, 8192]; odd: a square gemv's, in [32, 1024]"""
    g = torch.Generator().manual_seed(500)
    u = torch.rand(case["count"], generator=g, dtype=torch.float64).tolist()
    return [int(round(math.exp(math.log(64) + t * math.log(128)))) if i % 2 == 0 else
            int(round(math.exp(math.log(32) + t * math.log(32)))) for i, t in enumerate(u)]


def _doubles(case, seed):
    """the doubles that the inputs are made from, by name"""
    g, op, e = _gen(seed), case["op"], case.get("e")
    if op == "dot":
        size = (case["n"] - 1) * case["inc"] + 1
        return {"x": values(g, size, e), "y": values(g, size, e)}
    if op == "axpy":
        return {"x": values(g, (case["n"] - 1) * case["incx"] + 1, e),
                "y": values(g, (case["n"] - 1) * case["incy"] + 1, e), "alpha": values(g, 1, e)}
    if op == "gemv":
        m, n = case["m"], case["n"]
        lx, ly = (m, n) if case["trans"] else (n, m)
        return {"A": values(g, m * n, e), "x": values(g, lx, e), "y": values(g, ly, e), "alpha": values(g, 1, e)}
    if op in ("gemm", "mfma"):
        m, n, k = case["m"], case["n"], case["k"]
        return {"A": values(g, m * k, e), "B": values(g, k * n, e), "C": values(g, m * n, e), "alpha": values(g, 1, e)}
    if op == "spmv":
        return {"matrix": powerlaw(g, case["rows"]), "x": values(g, case["rows"], e)}
    if op == "cg":
        n = case["grid"] ** 2
        return {"matrix": grid_laplacian(case["grid"]), "b": values(g, n, 4)}
    ins, outs = 1, 0
    for i, s in enumerate(batch_sizes(case)):
        ins, outs = (ins + 2 * s, outs + 1) if i % 2 == 0 else (ins + s * s + s, outs + s)
    return {"in": values(g, ins, e), "out": values(g, outs, e)}


def prepare(case, seed):
    op, bits = case["op"], case["bits"]
    c = context(bits)
    d = _doubles(case, seed)
    s = {"op": op, "c": c, "L": c.L, "case": dict(case)}
    half = torch.full((1,), 0.5, dtype=torch.float64, device=DEV)
    if op == "dot":
        s["x"], s["y"], s["r"] = (Array(bits, d["x"].numel(), d["x"]), Array(bits, d["y"].numel(), d["y"]),
                                  Array(bits, 1))
        s["out"] = torch.empty(1, dtype=torch.float64, device=DEV)
    elif op == "axpy":
        for k in ("x", "y", "alpha"):
            s[k] = Array(bits, d[k].numel(), d[k])
    elif op in ("gemv", "gemm", "mfma"):
        for k in d:
            s[k] = Array(bits, d[k].numel(), d[k])
        s["beta"] = Array(bits, 1, half)  # a bounded update: repeated calls stay in range
        s["out"] = torch.empty(s["y" if op == "gemv" else "C"].size, dtype=torch.float64, device=DEV)
    elif op == "spmv":
        s["matrix"] = d["matrix"]
        s["csr"] = mp.Csr(d["matrix"][2].data_ptr(), d["matrix"][1].data_ptr(), d["matrix"][0].data_ptr())
        s["x"], s["y"] = Records(bits, case["rows"], d["x"]), Records(bits, case["rows"])
    elif op == "cg":
        n = case["grid"] ** 2
        s["matrix"], s["n"] = d["matrix"], n
        s["csr"] = mp.Csr(d["matrix"][2].data_ptr(), d["matrix"][1].data_ptr(), d["matrix"][0].data_ptr())
        s["b"], s["x"] = Records(bits, n, d["b"]), Records(bits, n)
        s["diag"] = torch.full((n,), 0.2, dtype=torch.float64, device=DEV)
        s["res"], s["its"] = (C.c_double * (case["iters"] + 1))(), C.c_int()
        s["out"] = torch.empty(n, dtype=torch.float64, device=DEV)
    else:
        a, o = Array(bits, d["in"].numel(), d["in"]), Array(bits, d["out"].numel(), d["out"])
        beta = Array(bits, 1, half)
        s["in"], s["res"], s["beta"], s["views"] = a, o, beta, []
        probs, i0, o0 = [], 1, 0
        al, be = a.view(0), beta.view(0)
        for i, z in enumerate(batch_sizes(case)):
            if i % 2 == 0:
                v = (a.view(i0), a.view(i0 + z), o.view(o0))
                probs.append(mp.dot_problem(z, *v, 1, 64))
                i0, o0 = i0 + 2 * z, o0 + 1
            else:
                v = (a.view(i0), a.view(i0 + z * z), o.view(o0))
                probs.append(mp.gemv_problem(mp.NO_TRANS, z, z, al, v[0], z, v[1], be, v[2], 8))
                i0, o0 = i0 + z * z + z, o0 + z
            s["views"].append(v)
        s["plan"] = mp.Batch(c, probs)
        s["out"] = torch.empty(o.size, dtype=torch.float64, device=DEV)
    return s


# ---------------------------------------------------------------- one pass
def run(s):
    op, c, L, k = s["op"], s["c"], s["L"], s["case"]
    if op == "dot":
        mp.check(L.mpres_dot(c.h, k["n"], s["x"].ref, k["inc"], s["y"].ref, k["inc"], s["r"].ref, k["grid"], k["block"],
                             None, 0, None))
        mp.check(L.mpres_array_get_d(c.h, 1, s["r"].ref, s["out"].data_ptr(), None))
        return {"r": s["r"].fields(), "double": s["out"]}
    if op == "axpy":
        mp.check(L.mpres_axpy(c.h, k["n"], s["alpha"].ref, s["x"].ref, k["incx"], s["y"].ref, k["incy"], None))
        return {"y": s["y"].fields()}
    if op == "gemv":
        mp.check(L.mpres_gemv(c.h, mp.TRANS if k["trans"] else mp.NO_TRANS, k["m"], k["n"], s["alpha"].ref, s["A"].ref,
                              k["m"], s["x"].ref, 1, s["beta"].ref, s["y"].ref, 1, k["block"], None, 0, None))
        mp.check(L.mpres_array_get_d(c.h, s["y"].size, s["y"].ref, s["out"].data_ptr(), None))
        return {"y": s["y"].fields(), "double": s["out"]}
    if op in ("gemm", "mfma"):
        f = L.mpres_gemm if op == "gemm" else L.mpres_gemm_mfma
        ta, tb = k.get("ta", False), k.get("tb", False)
        mp.check(f(c.h, mp.TRANS if ta else mp.NO_TRANS, mp.TRANS if tb else mp.NO_TRANS, k["m"], k["n"], k["k"],
                   s["alpha"].ref, s["A"].ref, k["k"] if ta else k["m"], s["B"].ref, k["n"] if tb else k["k"],
                   s["beta"].ref, s["C"].ref, k["m"], None, 0, None))
        mp.check(L.mpres_array_get_d(c.h, s["C"].size, s["C"].ref, s["out"].data_ptr(), None))
        return {"C": s["C"].fields(), "double": s["out"]}
    if op == "spmv":
        mp.check(L.mpres_spmv_csrv(c.h, k["rows"], C.byref(s["csr"]), k["tpr"], s["x"].ptr, s["y"].ptr, None))
        return {"y": s["y"].fields()}
    if op == "cg":
        s["x"].mem.zero_()  # the initial guess
        mp.check(L.mpres_cg_csr(c.h, s["n"], C.byref(s["csr"]), s["b"].ptr, 0.0, k["iters"], s["x"].ptr,
                                s["diag"].data_ptr(), s["res"], C.byref(s["its"]), 64, 128, None, 0, None))
        mp.check(L.mpres_get_d(c.h, s["n"], s["x"].ptr, s["out"].data_ptr(), None))
        return {"x": s["x"].fields(), "double": s["out"], "residuals": list(s["res"]), "iterations": s["its"].value}
    s["plan"].run()
    mp.check(L.mpres_array_get_d(c.h, s["res"].size, s["res"].ref, s["out"].data_ptr(), None))
    return {"results": s["res"].fields(), "double": s["out"]}


# ---------------------------------------------------------------- what a pass cannot do without
def work(case):
    """every operand read once, every result written once; a multiply and an add per residue and term"""
    op, n = case["op"], MODULI[case["bits"]]
    S = 4 * n + 40
    if op == "dot":
        return {"bytes": (2 * case["n"] + 1) * S, "flops": 2 * case["n"] * n}
    if op == "axpy":
        return {"bytes": (3 * case["n"] + 1) * S, "flops": 2 * case["n"] * n}
    if op == "gemv":
        a, b = case["m"], case["n"]
        lx, ly = (a, b) if case["trans"] else (b, a)
        return {"bytes": (a * b + lx + 2 * ly + 2) * S + 8 * ly, "flops": 2 * a * b * n}
    if op in ("gemm", "mfma"):
        a, b, k = case["m"], case["n"], case["k"]
        return {"bytes": (a * k + k * b + 2 * a * b + 2) * S + 8 * a * b, "flops": 2 * a * b * k * n}
    if op == "spmv":
        r, nnz = case["rows"], 15.9 * case["rows"]
        return {"bytes": 12 * nnz + 4 * (r + 1) + 2 * r * S, "flops": 2 * nnz * n}
    if op == "cg":
        g, it = case["grid"], case["iters"]
        r, nnz = g * g, 5 * g * g - 4 * g
        # per iteration: the matrix, x, r and p read and written, q written and read
        return {"bytes": it * (12 * nnz + 4 * (r + 1) + 8 * r * S) + 8 * r, "flops": it * 2 * (nnz + 5 * r) * n}
    fma = ins = outs = 0
    for i, z in enumerate(batch_sizes(case)):
        fma, ins, outs = (fma + z, ins + 2 * z, outs + 1) if i % 2 == 0 else (fma + z * z, ins + z * z + 2 * z, outs + z)
    return {"bytes": (ins + outs) * S + 8 * outs, "flops": 2 * fma * n}


# ---------------------------------------------------------------- the same in 64 bits
def exact(case, seed):
    op, d = case["op"], _doubles(case, seed)
    if op == "dot":
        x, y = d["x"][::case["inc"]], d["y"][::case["inc"]]
        return {"r": None, "double": torch.dot(x, y).reshape(1)}
    if op == "gemv":
        A = d["A"].view(case["n"], case["m"])  # column-major: row j of the view is column j
        prod = torch.mv(A, d["alpha"] * d["x"]) if case["trans"] else torch.mv(A.t(), d["alpha"] * d["x"])
        return {"y": None, "double": prod + 0.5 * d["y"]}
    if op in ("gemm", "mfma"):
        m, n, k = case["m"], case["n"], case["k"]
        A = d["A"].view(m, k) if case.get("ta") else d["A"].view(k, m).t()
        B = d["B"].view(k, n) if case.get("tb") else d["B"].view(n, k).t()
        Cm = d["alpha"] * torch.mm(A.contiguous(), B.contiguous()) + 0.5 * d["C"].view(n, m).t()
        return {"C": None, "double": Cm.t().contiguous().reshape(-1)}
    if op == "cg":
        irp, ja, vals = d["matrix"]
        n, b = case["grid"] ** 2, d["b"]
        A = torch.sparse_csr_tensor(irp.long(), ja.long(), vals, (n, n)).to_dense() if n <= 4096 else \
            torch.sparse_csr_tensor(irp.long(), ja.long(), vals, (n, n))
        x, r = torch.zeros_like(b), b.clone()
        z = 0.2 * r
        p, rho = z.clone(), torch.dot(r, z)
        for _ in range(case["iters"]):
            q = A @ p
            a = rho / torch.dot(p, q)
            x, r = x + a * p, r - a * q
            z = 0.2 * r
            rho, old = torch.dot(r, z), rho
            p = z + (rho / old) * p
        return {"x": None, "double": x, "residuals": None, "iterations": None}
    if op == "batch":
        a, o, al = d["in"], d["out"], d["in"][0]
        got, i0, o0 = [], 1, 0
        for i, z in enumerate(batch_sizes(case)):
            if i % 2 == 0:
                got.append(torch.dot(a[i0:i0 + z], a[i0 + z:i0 + 2 * z]).reshape(1))
                i0, o0 = i0 + 2 * z, o0 + 1
            else:
                A = a[i0:i0 + z * z].view(z, z).t()
                got.append(al * torch.mv(A, a[i0 + z * z:i0 + z * z + z]) + 0.5 * o[o0:o0 + z])
                i0, o0 = i0 + z * z + z, o0 + z
        return {"results": None, "double": torch.cat(got)}
    return None  # axpy and SpMV leave their results in multiple precision
