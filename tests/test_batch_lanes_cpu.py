"""The lanes a batch plan over 16 moduli chooses: one a number where gemvs with more chains than a
workgroup has lanes are nearly all of the work, not for one large gemv among many dots."""
import ctypes as C
import os
import subprocess

import pytest

from test_batch_cpu import mp

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def emu(tmp_path_factory):
    out = tmp_path_factory.mktemp("rule") / "lib.so"
    cmd = ["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-I", os.path.join(ROOT, "tests", "host", "emu"),
           os.path.join(ROOT, "tests", "host", "batch_rule_emu.cpp"), "-o", str(out)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return C.CDLL(str(out))


def gemv(m, n, block3, trans=mp.NO_TRANS):
    return mp.BatchProblem(op=mp.BATCH_GEMV, trans=trans, m=m, n=n, lda=m, incx=1, incy=1, block3=block3)


def dot(n):
    return mp.BatchProblem(op=mp.BATCH_DOT, n=n, incx=1, incy=1, grid3=1, block3=64)


@pytest.mark.parametrize("probs,want", [
    ([], 0), ([dot(8192)] * 3, 0), ([gemv(200, 200, 8)] * 4, 1),
    ([gemv(32, 900, 8)], 0), ([gemv(33, 900, 8)], 1),  # 256 and 264 chains
    ([gemv(900, 32, 8, mp.TRANS)], 0), ([gemv(900, 33, 8, mp.TRANS)], 1),
    ([dot(1700)] * 512 + [gemv(200, 200, 8)], 0),  # the costliest problem is the gemv
    ([dot(1000)] * 40 + [gemv(280, 1000, 8)], 0), ([dot(1000)] * 40 + [gemv(281, 1000, 8)], 1),  # 7/8
    ([gemv(0, 5, 8), dot(0)], 0)])
def test_one_lane(emu, probs, want):
    arr = (mp.BatchProblem * max(1, len(probs)))(*probs)
    assert emu.emu_batch_one_lane(arr, len(probs)) == want
