"""Moduli that the integer arithmetic cannot take are refused when a set's constants are computed: 3 m must
stay below 2^32, and the moduli of a set have one bit length."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def odd_coprime(start, n):
    """n pairwise coprime odd numbers from start on"""
    import math

    out = []
    while len(out) < n:
        if start % 2 and all(math.gcd(start, m) == 1 for m in out):
            out.append(start)
        start += 1
    return out


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = tmp_path_factory.mktemp("consts") / "lib.so"
    cmd = ["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off", "-I",
           os.path.join(ROOT, "tests", "host", "emu"), os.path.join(ROOT, "tests", "host", "consts_check.cpp"),
           os.path.join(ROOT, "mpres-blas_amd", "csrc", "consts.cpp"), "-o", str(out)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return C.CDLL(str(out))


@pytest.mark.parametrize("n", [8, 16, 32])
@pytest.mark.parametrize("start,ok", [(1 << 27, True), (1283742825, True), (1431655000 - 4000, True),
                                      (1431655766, False), (1500000001, False), (2147480001, False)])
def test_largest_modulus(lib, n, start, ok):
    m = odd_coprime(start, n)
    prod = 1
    for v in m:
        prod *= v
    assert bool(lib.check_set(n, prod.bit_length() - 1, (C.c_int * 32)(*m))) == ok


def test_one_bit_length(lib):
    m = odd_coprime((1 << 27) - 9, 8)
    prod = 1
    for v in m:
        prod *= v
    assert not lib.check_set(8, prod.bit_length() - 1, (C.c_int * 32)(*m))
