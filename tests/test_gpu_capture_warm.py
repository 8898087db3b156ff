"""Products captured into a graph by a context whose other products have left the
workspaces that they need, but of another shape: capturing allocates nothing, and what
the graph uses stays where it is.  Replays between other work of the context, bit-exact
against the oracle."""
import ctypes

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

RNS = 3


def hip():
    with open("/proc/self/maps") as maps:  # the HIP runtime that the library uses
        return ctypes.CDLL(next(line.split()[-1] for line in maps if "libamdhip64" in line))


def product(g, ctx, m, n, k, p, seed, **how):
    """C = A B on the context, its inputs and the call."""
    Ah, Bh = O.draw_matrix(m, k, p, seed), O.draw_matrix(k, n, p, seed + 1)
    A, B = g.CuModMatrix(Ah, p, elem_type=np.float64, ctx=ctx), g.CuModMatrix(Bh, p, elem_type=np.float64, ctx=ctx)
    C = g.zeros(np.float64, m, n, p, ctx=ctx)
    return C, (lambda: g.mul_(C, A, B, **how)), lambda: O.gemm(Ah, Bh, p)


# before, captured and afterwards: the planes and slices of the first are the largest,
# the rows or row blocks of the last
@pytest.mark.parametrize("name,p,before,inside,after", [
    ("multi-modular", 2 ** 26 - 5, (600, 600, 5000, RNS), (1500, 200, 40, RNS), (3000, 100, 30, RNS)),
    ("multi-modular", 65521, (600, 600, 4000, RNS), (1500, 200, 900, RNS), (3000, 100, 300, RNS)),
    ("vector", 65521, (512, 512, 4096, 1), (3000, 1, 2000, None), (20000, 1, 600, None)),
    ("vector", 2 ** 26 - 5, (512, 512, 4096, 1), (1001, 1, 515, None), (20000, 1, 600, None)),
])
def test_capture_after_other_shapes(gffm, name, p, before, inside, after):
    g, runtime = gffm, hip()
    print(f"capture {name} {inside} after {before}, p={p}", flush=True)
    ctx = g.Context()

    def make(shape, seed):
        m, n, k, form = shape
        return product(g, ctx, m, n, k, p, seed, **({} if form is None else {"form": form}))

    C0, run0, ref0 = make(before, 91)
    C1, run1, ref1 = make(inside, 93)
    C2, run2, ref2 = make(after, 95)
    run0()
    ctx.synchronize()
    assert np.array_equal(g.Array(C0).astype(np.int64), ref0())
    stream = ctypes.c_void_p(ctx.lib.modp_stream(ctx.h))
    graph, replay = ctypes.c_void_p(), ctypes.c_void_p()
    assert runtime.hipStreamBeginCapture(stream, 1) == 0
    try:
        run1()
    finally:
        status = runtime.hipStreamEndCapture(stream, ctypes.byref(graph))
    assert status == 0
    assert runtime.hipGraphInstantiate(ctypes.byref(replay), graph, None, None, ctypes.c_size_t(0)) == 0
    expect1, expect2 = ref1(), ref2()
    for i in range(3):
        C1.data.zero()
        assert runtime.hipGraphLaunch(replay, stream) == 0
        ctx.synchronize()
        assert np.array_equal(g.Array(C1).astype(np.int64), expect1), i
        run2()  # more rows, in planes and slices that are there
        run1()
        ctx.synchronize()
        assert np.array_equal(g.Array(C1).astype(np.int64), expect1), i
        assert np.array_equal(g.Array(C2).astype(np.int64), expect2), i
    assert runtime.hipGraphExecDestroy(replay) == 0 and runtime.hipGraphDestroy(graph) == 0
