"""Reductions over 8 moduli on data whose sums need no rounding for long runs, or now and then, where the
positional chains go on in residues (quads and single lanes), bit for bit against the oracle."""
import ctypes as C
import importlib.util
import os

import numpy as np
import pytest

import pyoracle as po
from test_quiet_cpu import KINDS, values

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
D = po.POLICY_D


def _load_mpres():
    spec = importlib.util.spec_from_file_location("mpres", os.path.join(ROOT, "mpres-blas_amd", "mpres.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


mp = _load_mpres()


@pytest.mark.parametrize("name", ["8_2double", "8_32bit"])
@pytest.mark.parametrize("kind", KINDS)
def test_quiet_reductions(name, kind):
    c, o = mp.Context(name), po.Oracle(name)
    L = c.L
    # quads: 12, 100 and 1600 terms a chain
    for n, g3, b3 in ((64 * 12, 8, 8), (64 * 100, 8, 8), (1600, 1, 1)):
        print(f"[case] quiet dot {name} {kind} {n} {g3}x{b3}", flush=True)
        xd, yd = values(kind, n, 1), values(kind, n, 2)
        x, y, r = c.array_set_d(xd), c.array_set_d(yd), c.array(1)
        mp.check(L.mpres_dot(c.h, n, C.byref(x), 1, C.byref(y), 1, C.byref(r), g3, b3, None, 0, None))
        assert c.array_to_host(r, 1).tobytes() == o.dot(o.set_d(xd, D), o.set_d(yd, D), g3, b3, D).tobytes()
    # quads, and a lane a chain (2100 * 32 chains)
    for trans, m, n, b3 in ((False, 65, 130, 2), (True, 130, 65, 2), (False, 2100, 320, 32)):
        print(f"[case] quiet gemv {name} {kind} {trans} {m}x{n} b3={b3}", flush=True)
        lx, ly = (m, n) if trans else (n, m)
        A, x, y = values(kind, m * n, 3), values(kind, lx, 4), values(kind, ly, 5)
        dA, dx, dy, da, db = (c.array_set_d(v) for v in (A, x, y, [1.0], [-1.0]))
        mp.check(L.mpres_gemv(c.h, mp.TRANS if trans else mp.NO_TRANS, m, n, C.byref(da), C.byref(dA), m, C.byref(dx), 1,
                              C.byref(db), C.byref(dy), 1, b3, None, 0, None))
        want = o.gemv(trans, m, n, o.set_d([1.0], D), o.set_d(A, D), m, o.set_d(x, D), o.set_d([-1.0], D),
                      o.set_d(y, D), b3, D)
        assert c.array_to_host(dy, ly).tobytes() == want.tobytes()
    m, n, k = 33, 20, 90
    print(f"[case] quiet gemm {name} {kind}", flush=True)
    A, B, Cm = (o.set_d(values(kind, q, s), D) for s, q in ((6, m * k), (7, k * n), (8, m * n)))
    al, be = o.set_d([1.0], D), o.set_d([-1.0], D)
    dA, dB, dC, da, db = (c.array_from_host(v) for v in (A, B, Cm, al, be))
    mp.check(L.mpres_gemm(c.h, mp.NO_TRANS, mp.NO_TRANS, m, n, k, C.byref(da), C.byref(dA), m, C.byref(dB), k,
                          C.byref(db), C.byref(dC), m, None, 0, None))
    want = o.gemm(m, n, k, al, A, m, B, k, be, Cm, m, D)
    assert c.array_to_host(dC, m * n).tobytes() == want.tobytes()
    c.close()


@pytest.mark.parametrize("name", ["16_4double", "32_8double"])
def test_sparse_gemm(name):
    """split-form gemm on sparse operands with zeros of both signs: entries whose every product is zero"""
    c, o, r = mp.Context(name), po.Oracle(name), np.random.default_rng(5)
    for m, n, k in ((64, 20, 17), (70, 65, 33)):
        print(f"[case] sparse gemm {name} {m}x{n}x{k}", flush=True)
        A, B, Cm = (o.set_d(np.where(r.uniform(0, 1, q) < 0.1, r.standard_normal(q), r.choice([0.0, -0.0], q)), D)
                    for q in (m * k, k * n, m * n))
        al, be = o.set_d([1.5], D), o.set_d([-1.0], D)
        dA, dB, dC, da, db = (c.array_from_host(v) for v in (A, B, Cm, al, be))
        mp.check(c.L.mpres_gemm(c.h, mp.NO_TRANS, mp.NO_TRANS, m, n, k, C.byref(da), C.byref(dA), m, C.byref(dB), k,
                                C.byref(db), C.byref(dC), m, None, 0, None))
        want = o.gemm(m, n, k, al, A, m, B, k, be, Cm, m, D)
        assert c.array_to_host(dC, m * n).tobytes() == want.tobytes()
    c.close()
