"""Element kernels with one lane per number over 16 and 32 moduli, compiled for the CPU with g++,
against the oracle bit for bit: operands that are doubles, full ones (every product rounds), and
sums that cancelled exactly (no residues left, bounds that are not zero). Modular products, long
division and integer square root against Python's integers."""
import ctypes as C
import math
import os
import random
import subprocess

import numpy as np
import pytest

import gen
import pyoracle as po

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
D = po.POLICY_D
W = 16  # limbs of the integers in round_emu.cpp


@pytest.fixture(scope="module")
def emu(tmp_path_factory):
    out = tmp_path_factory.mktemp("round") / "libround.so"
    cmd = ["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off", "-DMPH_SP_TS=1", "-DMPH_SPW_T=1",
           "-I", os.path.join(ROOT, "tests", "host", "emu"), os.path.join(ROOT, "tests", "host", "round_emu.cpp"),
           os.path.join(ROOT, "mpres-blas_amd", "csrc", "consts.cpp"), "-o", str(out)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return C.CDLL(str(out))


def P(a):
    return a.ctypes.data_as(C.c_void_p)


@pytest.mark.parametrize("name", ["16_4double", "32_8double", "16_32bit"])
@pytest.mark.parametrize("kind", ["doubles", "full", "cancelled"])
def test_elements(emu, name, kind):
    o, sid, n = po.Oracle(name), po.set_names().index(name), 300
    xd, yd = gen.uexp(5, n, -40, 40), gen.uexp(6, n, -40, 40)
    xd[7] = yd[9] = 0.0
    x, y = o.set_d(xd, D), o.set_d(yd, D)
    if kind != "doubles":
        for _ in range(10):
            x = o.mul(o.mul(x, x, D), y, D)
            y = o.add(o.mul(y, y, D), x, D)
    if kind == "cancelled":
        z = x.copy()
        z["sign"] ^= 1
        x = o.add(o.mul(o.add(x, z, D), y, D), o.add(y, y, D), D)
    r = o.empty(n)
    a = x[:1].copy()
    for op, want in ((0, o.add(x, y, D)), (1, o.sub(x, y, D)), (2, o.mul(x, y, D)), (3, o.mul_d(x, yd, D)),
                     (4, o.vadd(x, y)), (5, o.axpy_v2(a, x, y, D)), (6, o.set_d(yd, D))):
        assert emu.emu_elem(sid, op, n, P(x), P(y), P(yd), P(r)) == 0
        bad = [i for i in range(n) if r[i].tobytes() != want[i].tobytes()]
        assert not bad, (op, bad[:5])


@pytest.mark.parametrize("name", ["8_2double", "16_4double", "32_8double", "16_32bit"])
def test_modular_products(emu, name):
    o, sid = po.Oracle(name), po.set_names().index(name)
    rng = random.Random(3)
    for i, m in enumerate(int(v) for v in o.moduli()):
        edge = [0, 1, 2, m // 2, m - 2, m - 1]
        a = np.array([u for u in edge for _ in edge] + [rng.randrange(m) for _ in range(2000)], dtype=np.int32)
        b = np.array(edge * len(edge) + [rng.randrange(m) for _ in range(2000)], dtype=np.int32)
        want = (a.astype(np.int64) * b.astype(np.int64)) % m
        for how in (0, 1):
            r = np.empty_like(a)
            emu.emu_mulmod(sid, how, i, len(a), P(a), P(b), P(r))
            assert (r == want).all(), (how, m)


def limbs(v):
    return np.array([(v >> (32 * i)) & 0xffffffff for i in range(W)], dtype=np.uint32)


def value(a):
    return sum(int(v) << (32 * i) for i, v in enumerate(a))


def test_long_division_and_root(emu):
    rng = random.Random(11)
    o = np.empty(W, dtype=np.uint32)
    for t in range(4000):
        L = rng.randint(1, 32 * W - 2)
        top = 1 << (L - 1)
        some = [top, 2 * top - 1, top | rng.randrange(top), top | (rng.randrange(top) & ~rng.randrange(top))]
        a, b, q = rng.choice(some), rng.choice(some), rng.randint(2, 32 * W)
        inexact = emu.emu_div(P(limbs(a)), P(limbs(b)), q, P(o))
        assert (value(o), bool(inexact)) == ((a << (q - 1)) // b, (a << (q - 1)) % b != 0), (a, b, q)
        s = rng.choice([0, 1, 2, (1 << rng.randint(1, 16 * W - 24)) - 1, rng.getrandbits(16 * W - 24) >> rng.randint(0, 200)])
        v = max(0, s * s + rng.choice([-1, 0, 1, s]))
        inexact = emu.emu_isqrt(P(limbs(v)), P(o))
        assert (value(o), bool(inexact)) == (math.isqrt(v), math.isqrt(v) ** 2 != v), v
