"""Rows per item chosen by a batch plan for wide gemvs (few outputs, long rows): the items' copies of
alpha * x stay within the allowance beyond those of items of the cap's rows, and block3 up to the
largest int is taken."""
import ctypes as C

import numpy as np
import pytest

import pyoracle as po
from test_batch_cpu import bemu, mp  # noqa: F401 (fixture)

SPARE = 256 << 20


@pytest.mark.parametrize("name,groups", [("8_2double", 32), ("16_4double", 256), ("32_8double", 32)])
@pytest.mark.parametrize("trans", [mp.NO_TRANS, mp.TRANS])
@pytest.mark.parametrize("shapes,block3", [([(512, 32768)], 32), ([(100, 1000000)], 256), ([(300, 60000)] * 40, 64),
                                           ([(64, 8192)], 256), ([(1024, 1024)], 8), ([(7, 2000000)], 2**31 - 1)])
def test_wide_gemvs(bemu, name, groups, trans, shapes, block3):  # noqa: F811
    n_mod, sid = po.Oracle(name).n, po.set_names().index(name)
    buf = (C.c_char * 4096)()  # layout reads no numbers
    p = C.addressof(buf)
    dims = [(ly, lx) if trans == mp.NO_TRANS else (lx, ly) for ly, lx in shapes]
    arr = (mp.BatchProblem * len(dims))(*[mp.BatchProblem(
        op=mp.BATCH_GEMV, trans=trans, m=m, n=n, lda=m, incx=1, incy=1, block3=block3, alpha=p, A=p, x=p, beta=p, y=p)
        for m, n in dims])

    def layout(grp):
        out, wsb, cap = np.zeros((100000, 6), np.int64), C.c_longlong(), 100000
        cnt = bemu.emu_batch_auto(sid, arr, len(dims), 128, grp, out.ctypes.data_as(C.c_void_p), cap, C.byref(wsb))
        assert 0 < cnt <= cap
        return out[:cnt], wsb.value

    (fine, ws), (coarse, least) = layout(groups), layout(0)
    assert least <= ws <= least + SPARE + 256 * len(fine)
    assert sum(b - a for *_, a, b, _ in fine) == sum(ly for ly, _ in shapes)
    assert (fine[:, 4] - fine[:, 3]).max() <= 128 and (fine[:, 4] > fine[:, 3]).all()
