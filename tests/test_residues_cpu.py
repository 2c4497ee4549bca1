"""Stored residues outside [0, m), as host arithmetic leaves them (a little below zero, m or a little
above it) and as a caller may store them (any int of the residue's class): the kernels, compiled
for the CPU with g++, must give what they give for the same numbers with residues in [0, m)."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import gen
import pyoracle as po

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
D = po.POLICY_D


def build(tmp_path_factory, src):
    out = tmp_path_factory.mktemp(src) / "lib.so"
    cmd = ["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off", "-pthread", "-DMPH_SP_TS=1", "-DMPH_SPW_T=1",
           "-I", os.path.join(ROOT, "tests", "host", "emu"), os.path.join(ROOT, "tests", "host", src + ".cpp"),
           os.path.join(ROOT, "mpres-blas_amd", "csrc", "consts.cpp"), "-o", str(out)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return C.CDLL(str(out))


@pytest.fixture(scope="module")
def elems(tmp_path_factory):
    return build(tmp_path_factory, "round_emu")


@pytest.fixture(scope="module")
def chains(tmp_path_factory):
    return build(tmp_path_factory, "pos_emu")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    return build(tmp_path_factory, "kernels_emu")


def P(a):
    return a.ctypes.data_as(C.c_void_p)


def operands(o, seed, n, kind):
    """numbers, and the same with residues outside [0, m). small: integers whose residues lie within 14
    of a modulus, stored as -14 .. -1 and m .. m + 1; wide: residues moved by multiples of m"""
    rng = np.random.default_rng(seed)
    m = o.moduli().astype(np.int64)
    if kind == "small":
        r = rng.integers(0, len(m), n)
        v = np.concatenate([np.arange(-14, 0), [0, 1]])[rng.integers(0, 16, n)]
        x = o.set_d(((m[r] * rng.integers(1, 2**20, n) + v) * rng.choice([-1.0, 1.0], n)).astype(np.float64), D)
        d = x["digits"].astype(np.int64)
        d = np.where(d >= m - 14, d - m, np.where(d <= 1, d + m, d))
    else:
        x = o.set_d(gen.uexp(seed, n, -20, 20), D)
        x = np.where(rng.integers(0, 2, n).astype(bool), o.mul(x, x, D), x)
        d = x["digits"].astype(np.int64) + m * rng.integers(-2, 3, x["digits"].shape)
        d = np.where(np.abs(d) < 2**31, d, x["digits"])
    y = x.copy()
    y["digits"] = d
    assert (y["digits"] != x["digits"]).any()
    return x, y


@pytest.mark.parametrize("name", ["16_4double", "32_8double", "16_32bit"])
@pytest.mark.parametrize("kind", ["small", "wide"])
def test_elements(elems, name, kind):
    o, sid, n = po.Oracle(name), po.set_names().index(name), 400
    (x, xr), (y, yr) = operands(o, 1, n, kind), operands(o, 2, n, kind)
    yd = gen.uexp(3, n, -20, 20)
    for op in range(6):  # add, sub, mul, mul_d, vadd, axpy_v2
        want, got = o.empty(n), o.empty(n)
        assert elems.emu_elem(sid, op, n, P(x), P(y), P(yd), P(want)) == 0
        assert elems.emu_elem(sid, op, n, P(xr), P(yr), P(yd), P(got)) == 0
        bad = [i for i in range(n) if got[i].tobytes() != want[i].tobytes()]
        assert not bad, (op, bad[:5])


@pytest.mark.parametrize("name", ["8_2double", "8_32bit"])
@pytest.mark.parametrize("kind", ["small", "wide"])
@pytest.mark.parametrize("mode", [0, 1])
def test_chains(chains, name, kind, mode):
    """the residue chain (0) and the positional chain (1; what it leaves, the residue chain does)"""
    o, sid, cnt, n = po.Oracle(name), po.set_names().index(name), 12, 40
    (x, xr), (y, yr) = operands(o, 1, cnt * n, kind), operands(o, 2, cnt * n, kind)
    want, got = o.empty(n), o.empty(n)
    chains.emu_pos_chains(sid, 0, P(x), P(y), cnt, n, P(want))
    assert chains.emu_pos_chains(sid, mode, P(xr), P(yr), cnt, n, P(got)) >= 0
    done = got["sign"] != 2
    assert got[done].tobytes() == want[done].tobytes()


@pytest.mark.parametrize("name", ["8_2double", "16_4double", "32_8double"])
@pytest.mark.parametrize("kind", ["small", "wide"])
def test_gemm(kernels, name, kind):
    o, sid = po.Oracle(name), po.set_names().index(name)
    m, n, k = 9, 7, 12
    (A, Ar), (B, Br), (Cm, Cr) = (operands(o, s, q, kind) for s, q in ((1, m * k), (2, k * n), (3, m * n)))
    (al, alr), (be, ber) = operands(o, 4, 40, kind), operands(o, 5, 40, kind)
    want = o.gemm_v2(0, 0, m, n, k, al, A, m, B, k, be, Cm, m, D)
    ws = o.empty(m * n)
    for split in (0, 1):
        got = Cr.copy()
        assert kernels.emu_gemm_v2(sid, 0, 0, m, n, k, P(alr), P(Ar), m, P(Br), k, P(ber), P(got), m, P(ws), split) == 0
        assert got.tobytes() == want.tobytes(), split
    if o.n > 8:
        got = Cr.copy()
        assert kernels.emu_gemm_v2_split(sid, 0, 0, m, n, k, P(alr), P(Ar), m, P(Br), k, P(ber), P(got), m, P(ws)) == 0
        assert got.tobytes() == want.tobytes()


@pytest.mark.parametrize("name", ["16_4double", "32_8double"])
@pytest.mark.parametrize("kind", ["small", "wide"])
def test_spmv(kernels, name, kind):
    o, sid, m = po.Oracle(name), po.set_names().index(name), 300
    irp, ja, as_ = gen.powerlaw_csr(81, m, kmax=200)
    x, xr = operands(o, 1, m, kind)
    want, got, counts = o.empty(m), o.empty(m), np.zeros(2, np.int32)
    assert kernels.emu_spmv_split(sid, m, P(irp), P(ja), P(as_), P(x), P(want), P(counts)) == 0
    assert kernels.emu_spmv_split(sid, m, P(irp), P(ja), P(as_), P(xr), P(got), P(counts)) == 0
    assert got.tobytes() == want.tobytes()
