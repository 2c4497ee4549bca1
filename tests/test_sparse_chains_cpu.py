"""The split-form gemm's scalar chains on absolute bounds (k_gemm_chain_abs) on sparse operands: entries
whose every product is zero, of either sign and with zero operands whose lower bound is -0, bit for
bit against the chains by fractions and exponents."""
import numpy as np
import pytest

import gen
import pyoracle as po
from test_chain_cpu import D, P, emu  # noqa: F401 (fixture)


@pytest.mark.parametrize("name", ["16_4double", "32_8double"])
@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 1)])
@pytest.mark.parametrize("nonzero", [0.0, 0.1, 0.4])
@pytest.mark.parametrize("minus", ["none", "some", "bounds"])
def test_zero_products(emu, name, ta, tb, nonzero, minus):  # noqa: F811
    o, sid = po.Oracle(name), po.set_names().index(name)
    m, n, k, r = 13, 9, 20, np.random.default_rng(3)
    zero = lambda q: -0.0 if minus == "none" else np.where(r.integers(0, 2, q) == 1, -0.0, 0.0)  # noqa: E731
    As, Bs = (np.where(r.uniform(0, 1, q) < nonzero, gen.uexp(s, q, -30, 30), zero(q)) for s, q in ((1, m * k), (2, k * n)))
    A, B = o.set_d(As, D), o.set_d(Bs, D)
    if minus == "bounds":  # zeros as a sum of zeros leaves them
        for X in (A, B):
            z = (X["eval"][:, 1]["frac"] == 0) & (r.integers(0, 3, len(X)) == 0)
            X["eval"]["frac"][z, 0] = -0.0
    w1, w2 = o.empty(m * n), o.empty(m * n)
    assert emu.emu_chain_abs(sid, ta, tb, m, n, k, P(A), k if ta else m, P(B), n if tb else k, P(w1), P(w2)) == 0
    assert w1.tobytes() == w2.tobytes()
    assert (w1["eval"][:, 1]["frac"] == 0).any()
