"""The positional reduction chains (mpres-blas_amd/csrc/pos.hpp), compiled for the CPU with g++,
against the residue chains they stand for: every field bit for bit, on operands that round
every step, that never round, that need drops and large shifts, on short significands, zeros
and full-precision operands; exact cancellations must be left to the residue kernels, and
every step by the exact rule must agree with the estimates."""
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
    out = tmp_path_factory.mktemp("pos") / "libpos.so"
    cmd = ["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off", "-DMPH_SP_TS=1", "-DMPH_SPW_T=1",
           "-I", os.path.join(ROOT, "tests", "host", "emu"), os.path.join(ROOT, "tests", "host", "pos_emu.cpp"),
           os.path.join(ROOT, "mpres-blas_amd", "csrc", "consts.cpp"), "-o", str(out)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return C.CDLL(str(out))


def P(a):
    return a.ctypes.data_as(C.c_void_p)


@pytest.mark.parametrize("name", ["8_2double", "8_32bit", "8_16bit", "16_4double", "16_32bit", "16_16bit"])
@pytest.mark.parametrize("span", [0, 8, 20, 60, 200])
@pytest.mark.parametrize("kind", ["plain", "zeros", "short", "full"])
def test_chains(emu, name, span, kind):
    o = po.Oracle(name)
    sid = po.set_names().index(name)
    cnt, chains = 40, 25
    xs, ys = gen.uexp(5, cnt * chains, -span, span), gen.uexp(6, cnt * chains, -span, span)
    if kind == "zeros":  # zero operands, and some chains with exactly cancelling terms
        xs[::5] = 0
        at = np.arange(2, cnt * chains, 7 * cnt)
        xs[at + 1], ys[at + 1] = xs[at], -ys[at]
    if kind == "short":
        xs = np.sign(xs) * np.exp2(np.round(np.log2(np.abs(xs) + 1e-300)))
        ys = np.round(ys * 4) / 4
    x, y = o.set_d(xs, D), o.set_d(ys, D)
    if kind == "full":
        x = o.mul(o.mul(x, y, D), o.mul(x, y, D), D)
        y = o.add(o.mul(y, y, D), x, D)
    want, fast, exact = o.empty(chains), o.empty(chains), o.empty(chains)
    assert emu.emu_pos_chains(sid, 0, P(x), P(y), cnt, chains, P(want)) == 0
    left = emu.emu_pos_chains(sid, 1, P(x), P(y), cnt, chains, P(fast))
    emu.emu_pos_chains(sid, 2, P(x), P(y), cnt, chains, P(exact))
    for got in (fast, exact):
        done = got["sign"] != 2
        assert got[done].tobytes() == want[done].tobytes()
    assert ((fast["sign"] == 2) == (exact["sign"] == 2)).all()
    if kind in ("plain", "full"):
        assert left == 0
    else:
        assert left < chains


@pytest.mark.parametrize("name", ["8_2double", "16_4double"])
def test_operands_outside_the_form(emu, name):
    """an evaluation far from its number, or a number above the working precision: the chain is left"""
    o = po.Oracle(name)
    sid = po.set_names().index(name)
    x, y = o.set_d(gen.uexp(1, 8, -8, 8), D), o.set_d(gen.uexp(2, 8, -8, 8), D)
    x["eval"][3, 1]["frac"] *= 1.25  # a wider evaluation than the form takes
    out = o.empty(2)
    assert emu.emu_pos_chains(sid, 1, P(x), P(y), 4, 2, P(out)) == 1
    assert out["sign"][0] == 2 and out["sign"][1] != 2
