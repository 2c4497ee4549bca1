"""Stored residues outside [0, m) on the GPU: every operation must give what it gives for the same
numbers with residues in [0, m) (tests/test_residues_cpu.py makes them)."""
import ctypes as C
import importlib.util
import os

import numpy as np
import pytest

import gen
import pyoracle as po
from test_residues_cpu import operands

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _load_mpres():
    spec = importlib.util.spec_from_file_location("mpres", os.path.join(ROOT, "mpres-blas_amd", "mpres.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


mp = _load_mpres()


@pytest.mark.parametrize("name", ["8_2double", "8_32bit", "16_4double", "32_8double"])
@pytest.mark.parametrize("kind", ["small", "wide"])
def test_residues_outside_the_range(name, kind):
    c, o = mp.Context(name), po.Oracle(name)
    L, n, m = c.L, 1500, 60
    pairs = [operands(o, s, q, kind) for s, q in ((1, n), (2, n), (3, m * m), (4, m * m), (5, m * m), (6, 40), (7, m * m * 16))]
    yd = mp.DevBuf(host=gen.uexp(8, n, -20, 20))
    irp, ja, as_ = gen.powerlaw_csr(9, n, kmax=300)
    keep = [mp.DevBuf(host=v) for v in (as_, ja, irp)]
    csr = mp.Csr(*(b.ptr for b in keep))

    def results(which):
        x, y, A, B, Cm, s, long = (p[which] for p in pairs)
        X, Y, S = (mp.DevBuf(host=v) for v in (x, y, s))
        out = {}

        def aos(what, count, call):
            print(f"[case] residues {name} {kind} {what} {which}", flush=True)
            r = mp.DevBuf(nbytes=count * c.size)
            mp.check(call(r))
            out[what] = r.to_numpy(np.uint8).tobytes()

        for lanes in (0, 1, 2, 4, 8, 16, 32):
            if lanes and not L.mpres_lanes_supported(c.h, lanes):
                continue
            c.set_lanes(mp.K_ELEM, lanes)
            c.set_lanes(mp.K_AXPY, lanes)
            for op in range(5):
                aos(("elem", op, lanes), n, lambda r: L.mpres_elementwise(c.h, op, n, X.ptr, (yd if op == 3 else Y).ptr,
                                                                          r.ptr, None))
            aos(("axpy_v2", lanes), n, lambda r: L.mpres_axpy_v2(c.h, n, S.ptr, X.ptr, Y.ptr, r.ptr, None))
        c.set_lanes(mp.K_ELEM, 0)
        c.set_lanes(mp.K_AXPY, 0)
        for mode in (0, 1):
            r = mp.DevBuf(nbytes=4 * n)
            mp.check(L.mpres_cmp(c.h, mode, n, X.ptr, Y.ptr, r.ptr, None))
            out["cmp", mode] = r.to_numpy(np.uint8).tobytes()
        aos("csr", n, lambda r: L.mpres_spmv_csr(c.h, n, C.byref(csr), X.ptr, r.ptr, None))
        aos("csrv", n, lambda r: L.mpres_spmv_csrv(c.h, n, C.byref(csr), 8, X.ptr, r.ptr, None))
        # the v1 calls
        a = {k: c.array_from_host(v) for k, v in (("x", x), ("y", y), ("A", A), ("B", B), ("s", s), ("long", long))}
        ref = {k: C.byref(v) for k, v in a.items()}

        def v1(what, r, count, rc):
            print(f"[case] residues {name} {kind} {what} {which}", flush=True)
            mp.check(rc)
            out[what] = c.array_to_host(r, count).tobytes()

        r = c.array_from_host(y)
        v1("axpy", r, n, L.mpres_axpy(c.h, n, ref["s"], ref["x"], 1, C.byref(r), 1, None))
        r = c.array(1)
        v1("dot", r, 1, L.mpres_dot(c.h, n, ref["x"], 1, ref["y"], 1, C.byref(r), 4, 8, None, 0, None))
        v1("long dot", r, 1, L.mpres_dot(c.h, len(long), ref["long"], 1, ref["long"], 1, C.byref(r), 16, 64, None, 0, None))
        v1("asum", r, 1, L.mpres_asum(c.h, n, ref["x"], 1, C.byref(r), 4, 8, None, 0, None))
        for t in (mp.NO_TRANS, mp.TRANS):
            r = c.array_from_host(y)
            v1(("gemv", t), r, m, L.mpres_gemv(c.h, t, m, m, ref["s"], ref["A"], m, ref["x"], 1, ref["s"], C.byref(r), 1, 8,
                                              None, 0, None))
        for what, f in (("gemm", L.mpres_gemm), ("mfma", L.mpres_gemm_mfma)):
            r = c.array_from_host(Cm)
            v1(what, r, m * m, f(c.h, mp.NO_TRANS, mp.NO_TRANS, m, m, m, ref["s"], ref["A"], m, ref["B"], m, ref["s"],
                                C.byref(r), m, None, 0, None))
        Ab, Bb, r = mp.DevBuf(host=A), mp.DevBuf(host=B), mp.DevBuf(host=Cm)
        mp.check(L.mpres_gemm_v2(c.h, mp.TRANS, mp.NO_TRANS, m, m, m, S.ptr, Ab.ptr, m, Bb.ptr, m, S.ptr, r.ptr, m, None, 0,
                                 None))
        out["gemm_v2"] = r.to_numpy(np.uint8).tobytes()
        r, d = c.array_from_host(y), c.array(1)
        b = mp.Batch(c, [mp.gemv_problem(mp.NO_TRANS, m, m, a["s"], a["A"], m, a["x"], a["s"], r, 8),
                         mp.dot_problem(n, a["x"], a["y"], d, 4, 8)])
        b.run()
        v1("batch gemv", r, m, 0)
        v1("batch dot", d, 1, 0)
        b.close()
        return out

    want, got = results(0), results(1)
    assert [k for k in want if want[k] != got[k]] == []
    c.close()
