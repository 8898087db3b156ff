"""Products of little depth where no workspace may be had: captured into a graph by a
context that has none yet, and with hardly any device memory left.  Bit-exact against
the oracle."""
import ctypes

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def hip():
    with open("/proc/self/maps") as maps:  # the HIP runtime that the library uses
        runtime = ctypes.CDLL(next(line.split()[-1] for line in maps if "libamdhip64" in line))
    runtime.hipMalloc.argtypes = [ctypes.c_void_p, ctypes.c_size_t]
    return runtime


@pytest.mark.parametrize("m,n,k", [(6000, 6000, 200), (8000, 7001, 128), (5100, 5100, 255)])
def test_capture_large(gffm, m, n, k):
    # large enough for the multi-modular form
    g, runtime, p = gffm, hip(), 2 ** 26 - 5
    print(f"capture {m}x{n}x{k}", flush=True)
    ctx = g.Context()
    Ah, Bh = O.draw_matrix(m, k, p, 71), O.draw_matrix(k, n, p, 72)
    A, B = g.CuModMatrix(Ah, p, elem_type=np.float64, ctx=ctx), g.CuModMatrix(Bh, p, elem_type=np.float64, ctx=ctx)
    C = g.zeros(np.float64, m, n, p, ctx=ctx)
    ctx.synchronize()
    stream = ctypes.c_void_p(ctx.lib.modp_stream(ctx.h))
    graph, run = ctypes.c_void_p(), ctypes.c_void_p()
    assert runtime.hipStreamBeginCapture(stream, 1) == 0
    try:
        g.mul_(C, A, B)
    finally:
        status = runtime.hipStreamEndCapture(stream, ctypes.byref(graph))
    assert status == 0
    assert runtime.hipGraphInstantiate(ctypes.byref(run), graph, None, None, ctypes.c_size_t(0)) == 0
    expect = O.gemm(Ah, Bh, p)
    for i in range(3):
        C.data.zero()
        assert runtime.hipGraphLaunch(run, stream) == 0
        ctx.synchronize()
        assert np.array_equal(g.Array(C).astype(np.int64), expect), i
        C.data.zero()
        g.mul_(C, A, B)  # with workspaces
        ctx.synchronize()
        assert np.array_equal(g.Array(C).astype(np.int64), expect), i
    assert runtime.hipGraphExecDestroy(run) == 0 and runtime.hipGraphDestroy(graph) == 0


@pytest.mark.parametrize("m,n,k,p", [(20000, 600, 200, 2 ** 26 - 5), (600, 40000, 255, 65521), (6000, 6000, 255, 2 ** 26 - 5)])
def test_little_memory(gffm, m, n, k, p):
    # room for less than the digit planes
    g, runtime = gffm, hip()
    print(f"little memory {m}x{n}x{k} p={p}", flush=True)
    ctx = g.Context()
    Ah, Bh = O.draw_matrix(m, k, p, 81), O.draw_matrix(k, n, p, 82)
    A, B = g.CuModMatrix(Ah, p, elem_type=np.float64, ctx=ctx), g.CuModMatrix(Bh, p, elem_type=np.float64, ctx=ctx)
    C = g.zeros(np.float64, m, n, p, ctx=ctx)
    X = g.rand(np.float64, 200, 200, p, seed=3, ctx=ctx)
    g.mul_(g.zeros(np.float64, 200, 200, p, ctx=ctx), X, X)  # (the plain form's code is on the device)
    ctx.synchronize()
    ctx.release_freed()
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    keep, ballast = 4 << 20, []
    try:
        for _ in range(4):  # (what is free is an estimate while much of it is)
            assert runtime.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
            if free.value <= keep + (4 << 20):
                break
            ballast.append(ctypes.c_void_p())
            if runtime.hipMalloc(ctypes.byref(ballast[-1]), free.value - keep) != 0:
                runtime.hipGetLastError()
                break
        print(f"{free.value} bytes left of {total.value}", flush=True)
        g.mul_(C, A, B)
        ctx.synchronize()
    finally:
        assert all([runtime.hipFree(x) == 0 for x in ballast if x.value])
    assert np.array_equal(g.Array(C).astype(np.int64), O.gemm(Ah, Bh, p))
    C.data.zero()
    g.mul_(C, A, B)  # with workspaces
    assert np.array_equal(g.Array(C).astype(np.int64), O.gemm(Ah, Bh, p))
