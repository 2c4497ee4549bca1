"""Choices that calls make when the caller leaves them open, bit for bit against the oracle: a batch plan's
geometry (lanes, rows per item), and the lanes of axpy over 16 moduli, where one lane of a pair does
a number that rounds again."""
import ctypes as C

import pytest

import gen
from test_gpu_parity import D, _batch_case, mp, orc

pytestmark = pytest.mark.gpu


def full(o, seed, n):
    """numbers whose products round"""
    x, y = o.set_d(gen.uexp(seed, n, -20, 20), D), o.set_d(gen.uexp(seed + 1, n, -20, 20), D)
    for _ in range(8):
        x = o.mul(x, y, D)
    return x


@pytest.mark.parametrize("name", ["8_2double", "16_4double", "32_8double"])
@pytest.mark.parametrize("large", [False, True])
def test_batch_geometry(name, large):
    """large: a gemv of full numbers is nearly all of the work (one lane a number at 16 moduli)"""
    c, o = mp.Context(name), orc(name)
    probs, keep, checks = _batch_case(c, o, name, 900)
    if large:
        m, n, b3 = 600, 450, 3
        Ar, xr, yr, ar, br = (full(o, s, q) for s, q in ((51, 4096), (53, n), (55, m), (57, 1), (59, 1)))
        Ar = Ar[(gen.np.arange(m * n) * 17) % 4096]
        A, x, y, al, be = (c.array_from_host(v) for v in (Ar, xr, yr, ar, br))
        probs.append(mp.gemv_problem(mp.NO_TRANS, m, n, al, A, m, x, be, y, b3))
        checks.append(("gemv", y, m, o.gemv(0, m, n, ar, Ar, m, xr, br, yr, b3, D), yr))
    print(f"[case] batch geometry {name} large={large}", flush=True)
    b = mp.Batch(c, probs)
    info = b.info()
    assert info["tuning"]["gemv_rows"] == 0
    if name.startswith("16_"):
        assert (info["tuning"]["lanes"] == 1) == large
    again = mp.Batch(c, probs, info["tuning"])
    assert again.info() == info
    for plan in (b, again):
        for kind, arr, cnt, want, reset in checks:
            if reset is not None:
                mp.check(c.L.mpres_array_host2device(c.h, C.byref(arr), reset.ctypes.data_as(C.c_void_p), cnt, None))
        plan.run()
        mp.synchronize()
        for i, (kind, arr, cnt, want, reset) in enumerate(checks):
            assert c.array_to_host(arr, cnt).tobytes() == want.tobytes(), (i, kind)
        plan.close()
    # a workspace for items of 128 rows only
    fixed = mp.BatchTuning(lanes=info["tuning"]["lanes"], wg_per_cu=4, gemv_rows=128)
    arr = (mp.BatchProblem * len(probs))(*probs)
    need = c.L.mpres_batch_workspace(c.h, arr, len(probs), C.byref(fixed))
    ws, h, used = mp.DevBuf(nbytes=need), C.c_void_p(), mp.BatchTuning()
    mp.check(c.L.mpres_batch_plan(c.h, arr, len(probs), None, ws.ptr, need, C.byref(h)))
    mp.check(c.L.mpres_batch_info(h, None, None, C.byref(used)))
    assert used.gemv_rows in (0, 128)
    mp.check(c.L.mpres_batch_destroy(h))
    c.close()


@pytest.mark.parametrize("n", [1, 257, 3001])
@pytest.mark.parametrize("lanes", [1, 2, 4, 16])
def test_axpy_16(n, lanes):
    c, o = mp.Context("16_4double"), orc("16_4double")
    c.set_lanes(mp.K_AXPY, lanes)
    print(f"[case] axpy 16 moduli n={n} lanes={lanes}", flush=True)
    x, y, a = full(o, 61, n), full(o, 63, n), full(o, 65, 1)
    d = o.set_d(gen.uexp(67, n, -20, 20), D)
    x[::3], y[1::3] = d[::3], d[1::3]  # numbers that round beside numbers that do not
    dx, dy, da = c.array_from_host(x), c.array_from_host(y), c.array_from_host(a)
    mp.check(c.L.mpres_axpy(c.h, n, C.byref(da), C.byref(dx), 1, C.byref(dy), 1, None))
    assert c.array_to_host(dy, n).tobytes() == o.axpy(a, x, y, D).tobytes()
    bx, by, ba, br = c.aos(x), c.aos(y), c.aos(a), c.aos(count=n)
    mp.check(c.L.mpres_axpy_v2(c.h, n, ba.ptr, bx.ptr, by.ptr, br.ptr, None))
    assert c.aos_to_host(br, n).tobytes() == o.axpy_v2(a, x, y, D).tobytes()
    c.close()
