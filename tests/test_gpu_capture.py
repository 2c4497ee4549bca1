"""A call captured into a HIP graph on the context's workspace pool, where the pool holds what the call needs
but not what it would like to have: the capture goes through, and every replay gives the eager result."""
import ctypes as C

import pytest

import gen
from test_gpu_parity import D, mp, orc

pytestmark = pytest.mark.gpu


def test_gemv_on_a_pool_that_would_do():
    c, e, o = mp.Context("8_2double"), mp.Context("8_2double"), orc("8_2double")
    H, m, b3 = mp.hip(), 64, 8
    st, graph, run = C.c_void_p(), C.c_void_p(), C.c_void_p()
    mp.hipchk(H.hipStreamCreate(C.byref(st)))
    A, x, y = (o.set_d(gen.uexp(s, n, -20, 20), D) for s, n in ((1, m * m), (2, m), (3, m)))
    al, be = o.set_d([1.25], D), o.set_d([0.5], D)

    def operands(ctx):
        return [ctx.array_from_host(v) for v in (al, A, x, be, y)]

    def gemv(ctx, a, stream):
        return ctx.L.mpres_gemv(ctx.h, mp.NO_TRANS, m, m, C.byref(a[0]), C.byref(a[1]), m, C.byref(a[2]), 1, C.byref(a[3]),
                                C.byref(a[4]), 1, b3, None, 0, stream)

    captured, eager = operands(c), operands(e)
    # a dot's partials bring the pool between the two sizes
    need, full = c.size * (m + m * b3 + m), c.L.mpres_gemv_workspace(c.h, mp.NO_TRANS, m, m, b3)
    g3, bb = 8, 71
    assert need <= c.L.mpres_dot_workspace(c.h, m, g3, bb) < full
    r = c.array(1)
    print("[case] capture on a smaller pool", flush=True)
    mp.check(c.L.mpres_dot(c.h, m, C.byref(captured[2]), 1, C.byref(captured[2]), 1, C.byref(r), g3, bb, None, 0, st))
    mp.hipchk(H.hipStreamSynchronize(st))
    mp.hipchk(H.hipStreamBeginCapture(st, 1))  # thread-local: allocations end it
    mp.check(gemv(c, captured, st))
    mp.hipchk(H.hipStreamEndCapture(st, C.byref(graph)))
    mp.hipchk(H.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)))
    for _ in range(3):
        mp.hipchk(H.hipGraphLaunch(run, st))
        mp.hipchk(H.hipStreamSynchronize(st))
        mp.check(gemv(e, eager, None))
        assert c.array_to_host(captured[4], m).tobytes() == e.array_to_host(eager[4], m).tobytes()
    mp.hipchk(H.hipGraphExecDestroy(run))
    mp.hipchk(H.hipGraphDestroy(graph))
    mp.hipchk(H.hipStreamDestroy(st))
    c.close()
    e.close()
