"""Positional reduction chains whose sums need no rounding for long runs (integers, doubles of few bits,
zeros), or now and then: they go on in residues and come back (pos_run in kernels_pos.hpp). Compiled for
the CPU with g++, bit for bit against the residue chain."""
import numpy as np
import pytest

import pyoracle as po
from test_pos_cpu import D, P, emu  # noqa: F401 (fixture)

KINDS = ["int", "pm1", "f32", "norm", "sparse", "mix", "rare"]


def values(kind, n, seed):
    r = np.random.default_rng(seed)
    few, some = r.uniform(0, 1, n) < 0.02, r.standard_normal(n)
    return {"int": lambda: r.integers(-1000, 1001, n).astype(np.float64),
            "pm1": lambda: r.choice([-1.0, 1.0], n),  # sums that cancel exactly
            "f32": lambda: some.astype(np.float32).astype(np.float64),
            "norm": lambda: some,
            "sparse": lambda: np.where(r.uniform(0, 1, n) < 0.9, 0.0, some),
            "mix": lambda: np.where(few, np.ldexp(some, r.integers(-60, 60, n)), r.integers(-50, 51, n)),
            "rare": lambda: np.where(few, some, r.integers(-5, 6, n))}[kind]()


@pytest.mark.parametrize("name", ["8_2double", "8_32bit"])
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("cnt", [7, 8, 9, 33, 700])  # around the first line, and past several
def test_quiet_chains(emu, name, kind, cnt):  # noqa: F811
    o, sid, chains = po.Oracle(name), po.set_names().index(name), 25
    x, y = o.set_d(values(kind, cnt * chains, 1), D), o.set_d(values(kind, cnt * chains, 2), D)
    want, got = o.empty(chains), o.empty(chains)
    assert emu.emu_pos_chains(sid, 0, P(x), P(y), cnt, chains, P(want)) == 0
    left = emu.emu_pos_chains(sid, 1, P(x), P(y), cnt, chains, P(got))
    done = got["sign"] != 2
    assert got[done].tobytes() == want[done].tobytes()
    assert left == (~done).sum() and (left == 0 or kind in ("pm1", "rare", "int"))
