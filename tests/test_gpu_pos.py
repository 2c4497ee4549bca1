"""The positional reduction chains on the GPU (8 moduli) where their dispatch changes, bit for bit
against the oracle: dots at the chain length from which they are used, chains that cancel or
whose operands are outside the form (left to the residue kernels), quads against single
lanes, and gemv and gemm with a workspace too small for the operands' records."""
import ctypes as C
import importlib.util
import os

import numpy as np
import pytest

import gen
import pyoracle as po

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
D = po.POLICY_D


def _load_mpres():
    spec = importlib.util.spec_from_file_location("mpres", os.path.join(ROOT, "mpres-blas_amd", "mpres.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


mp = _load_mpres()


@pytest.fixture(scope="module", params=["8_2double", "8_32bit"])
def ctx(request):
    c = mp.Context(request.param)
    yield c, po.Oracle(request.param)
    c.close()


# (n, grid, block): 7, 8 and 9 terms in the longest chain around the line; more chains than quads serve
@pytest.mark.parametrize("n,g3,b3", [(64 * 8 - 1, 8, 8), (64 * 8, 8, 8), (64 * 8 + 1, 8, 8), (600000, 1100, 64)])
@pytest.mark.parametrize("kind", ["plain", "cancel"])
def test_dot(ctx, n, g3, b3, kind):
    c, o = ctx
    print(f"[case] pos dot {c.set_name} {n} {g3}x{b3} {kind}", flush=True)
    xd, yd = gen.uexp(11, n, -20, 20), gen.uexp(12, n, -20, 20)
    if kind == "cancel":  # chain 0 cancels exactly after its second term
        xd[g3 * b3], yd[g3 * b3] = xd[0], -yd[0]
    x, y, r = c.array_set_d(xd), c.array_set_d(yd), c.array(1)
    mp.check(c.L.mpres_dot(c.h, n, C.byref(x), 1, C.byref(y), 1, C.byref(r), g3, b3, None, 0, None))
    want = o.dot(o.set_d(xd, D), o.set_d(yd, D), g3, b3, D)
    assert c.array_to_host(r, 1).tobytes() == want.tobytes()


@pytest.mark.parametrize("trans", [False, True])
@pytest.mark.parametrize("m,n,b3", [(5, 3, 8), (65, 130, 16), (2100, 40, 32)])
@pytest.mark.parametrize("small", [False, True])
def test_gemv_workspace(ctx, trans, m, n, b3, small):
    c, o = ctx
    print(f"[case] pos gemv {c.set_name} {m}x{n} b3={b3} trans={trans} small={small}", flush=True)
    lx, ly = (m, n) if trans else (n, m)
    A, x, y = gen.uexp(21, m * n, -20, 20), gen.uexp(22, lx, -20, 20), gen.uexp(23, ly, -20, 20)
    al, be = [1.25], [-0.75]
    dA, dx, dy = c.array_set_d(A), c.array_set_d(x), c.array_set_d(y)
    da, db = c.array_set_d(al), c.array_set_d(be)
    t = mp.TRANS if trans else mp.NO_TRANS
    need = c.size * (lx + ly * b3 + ly)  # without room for the records
    wsb = need if small else c.L.mpres_gemv_workspace(c.h, t, m, n, b3)
    assert wsb >= need
    ws = mp.DevBuf(nbytes=wsb)
    mp.check(c.L.mpres_gemv(c.h, t, m, n, C.byref(da), C.byref(dA), m, C.byref(dx), 1, C.byref(db), C.byref(dy), 1, b3,
                            ws.ptr, wsb, None))
    want = o.gemv(trans, m, n, o.set_d(al, D), o.set_d(A, D), m, o.set_d(x, D), o.set_d(be, D), o.set_d(y, D), b3, D)
    assert c.array_to_host(dy, ly).tobytes() == want.tobytes()


@pytest.mark.parametrize("small", [False, True])
@pytest.mark.parametrize("bad", [False, True])
def test_gemm_workspace(ctx, small, bad):
    c, o = ctx
    m, n, k = 33, 65, 70
    print(f"[case] pos gemm {c.set_name} small={small} bad={bad}", flush=True)
    A, B, Cm = (o.set_d(gen.uexp(s, q, -20, 20), D) for s, q in ((31, m * k), (32, k * n), (33, m * n)))
    if bad:  # an evaluation wider than the form takes: row 4's chains are left to the residue kernels
        A["eval"][4 + 2 * m, 1]["frac"] *= 1.25
    al, be = o.set_d([1.25], D), o.set_d([-0.75], D)
    dA, dB, dC, da, db = (c.array_from_host(v) for v in (A, B, Cm, al, be))
    need = (m * n * c.size + 255) // 256 * 256
    wsb = need if small else c.L.mpres_gemm_workspace(c.h, m, n, k)
    ws = mp.DevBuf(nbytes=wsb)
    mp.check(c.L.mpres_gemm(c.h, mp.NO_TRANS, mp.NO_TRANS, m, n, k, C.byref(da), C.byref(dA), m, C.byref(dB), k,
                            C.byref(db), C.byref(dC), m, ws.ptr, wsb, None))
    want = o.gemm(m, n, k, al, A, m, B, k, be, Cm, m, D)
    assert c.array_to_host(dC, m * n).tobytes() == want.tobytes()
