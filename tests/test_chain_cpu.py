"""The split-form gemm's scalar chains on absolute bounds (k_gemm_chain_abs), compiled for the CPU
with g++, against the chains by fractions and exponents (k_gemm_chain): every entry's sign,
exponent and evaluation, or its REDO mark, bit for bit - on ordinary operands, on sums near the
rounding threshold, zeros, exact cancellations, and operands outside the form's range."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import gen
import pyoracle as po

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
D = po.POLICY_D


@pytest.fixture(scope="module")
def emu(tmp_path_factory):
    out = tmp_path_factory.mktemp("chain") / "libchain.so"
    cmd = ["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off", "-DMPH_SP_TS=1", "-DMPH_SPW_T=1",
           "-I", os.path.join(ROOT, "tests", "host", "emu"), os.path.join(ROOT, "tests", "host", "chain_emu.cpp"),
           os.path.join(ROOT, "mpres-blas_amd", "csrc", "consts.cpp"), "-o", str(out)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return C.CDLL(str(out))


def P(a):
    return a.ctypes.data_as(C.c_void_p)


@pytest.mark.parametrize("name", ["16_4double", "32_8double", "16_32bit"])
@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 0), (0, 1)])
@pytest.mark.parametrize("span,kind", [(8, "plain"), (30, "plain"), (53, "plain"), (150, "plain"), (400, "plain"),
                                       (20, "zeros"), (20, "full")])
def test_chain_abs(emu, name, ta, tb, span, kind):
    o = po.Oracle(name)
    sid = po.set_names().index(name)
    m, n, k = 11, 7, 37
    As, Bs = gen.uexp(41, m * k, -span, span), gen.uexp(42, k * n, -span, span)
    if kind == "zeros":
        As[::4], Bs[::7] = 0.0, -0.0
        As[:3 * (k if ta else 1)] = 0.0
    A, B = o.set_d(As, D), o.set_d(Bs, D)
    if kind == "full":
        A, B = o.mul(A, A, D), o.mul(o.mul(B, B, D), B, D)
    w1, w2 = o.empty(m * n), o.empty(m * n)
    unusual = emu.emu_chain_abs(sid, ta, tb, m, n, k, P(A), k if ta else m, P(B), n if tb else k, P(w1), P(w2))
    assert unusual >= 0 and (unusual > 0) == (span > 200)
    assert w1.tobytes() == w2.tobytes()
    if span == 8:
        assert (w1["sign"] != 2).all()
