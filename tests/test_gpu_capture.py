"""Products captured into a graph by a context that has no workspaces yet: the ones
that are small enough to need none.  Replays between other work of the context,
bit-exact against the oracle."""
import ctypes

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def hip():
    with open("/proc/self/maps") as maps:  # the HIP runtime that the library uses
        return ctypes.CDLL(next(line.split()[-1] for line in maps if "libamdhip64" in line))


@pytest.mark.parametrize("et,p", [(np.float64, 65521), (np.float64, 2 ** 26 - 5), (np.float32, 11)])
@pytest.mark.parametrize("m,n,k", [(64, 64, 64), (48, 40, 56), (700, 500, 100), (1501, 1203, 255), (300, 280, 47), (1000, 1, 500), (2, 1, 512)])
def test_capture_without_workspaces(gffm, m, n, k, et, p):
    g, runtime = gffm, hip()
    print(f"capture {m}x{n}x{k} p={p}", flush=True)
    ctx = g.Context()
    Ah, Bh = O.draw_matrix(m, k, p, 71), O.draw_matrix(k, n, p, 72)
    A, B = g.CuModMatrix(Ah, p, elem_type=et, ctx=ctx), g.CuModMatrix(Bh, p, elem_type=et, ctx=ctx)
    C = g.zeros(et, m, n, p, ctx=ctx)
    ctx.synchronize()
    stream = ctypes.c_void_p(ctx.lib.modp_stream(ctx.h))
    graph, run = ctypes.c_void_p(), ctypes.c_void_p()
    square = m == n == k  # then over its first operand
    C = A if square else C
    assert runtime.hipStreamBeginCapture(stream, 1) == 0
    try:
        g.mul_(C, A, B)
    finally:
        status = runtime.hipStreamEndCapture(stream, ctypes.byref(graph))
    assert status == 0
    assert runtime.hipGraphInstantiate(ctypes.byref(run), graph, None, None, ctypes.c_size_t(0)) == 0
    X = g.rand(np.float64, 900, 900, 65521, seed=9, ctx=ctx)
    for i in range(3):
        if not square:
            C.data.zero()
        assert runtime.hipGraphLaunch(run, stream) == 0
        ctx.synchronize()
        assert np.array_equal(g.Array(C).astype(np.int64), O.gemm(Ah, Bh, p)), i
        Ah = O.gemm(Ah, Bh, p) if square else Ah
        Y = X * X  # workspaces come and grow in between
        ctx.synchronize()
        del Y
    assert runtime.hipGraphExecDestroy(run) == 0 and runtime.hipGraphDestroy(graph) == 0
