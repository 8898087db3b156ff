"""Reduced echelon forms of tall matrices with less device memory left than the digit
planes of the trailing updates take: equal to those with memory."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,rank,p", [(120000, 600, 600, 65521), (60000, 700, 600, 2 ** 26 - 5), (150000, 520, 300, 11)])
def test_tall_with_little_memory(gffm, m, n, rank, p):
    g = gffm
    print(f"little memory: rref {m}x{n} rank {rank} p={p}", flush=True)
    with open("/proc/self/maps") as maps:  # the HIP runtime that the library uses
        runtime = ctypes.CDLL(next(line.split()[-1] for line in maps if "libamdhip64" in line))
    runtime.hipMalloc.argtypes = [ctypes.c_void_p, ctypes.c_size_t]
    A = g.rand(np.float64, m, rank, p, seed=1) * g.rand(np.float64, rank, n, p, seed=2)
    whole, pivots, r = g.rref_full(A)
    expect = g.Array(whole)
    assert r == rank and np.array_equal(expect[:rank, np.asarray(pivots) - 1], np.eye(rank))
    assert not expect[rank:].any()
    ctx = g.Context()
    B = g.CuModMatrix(g.Array(A), p, elem_type=np.float64, ctx=ctx)
    del A, whole
    g.rref(g.rand(np.float64, 2000, 300, p, seed=3, ctx=ctx))
    ctx.synchronize()
    ctx.release_freed()
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    # the result, the elimination's own copy, row positions, and 10 MB
    keep, ballast = 8 * (m + 32) * (n + 32) + 4 * (m + 64) * n + 8 * m + (10 << 20), []
    try:
        for _ in range(4):  # (what is free is an estimate while much of it is)
            assert runtime.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
            if free.value <= keep + (4 << 20):
                break
            ballast.append(ctypes.c_void_p())
            assert runtime.hipMalloc(ctypes.byref(ballast[-1]), free.value - keep) == 0
        print(f"{free.value} bytes left of {total.value}", flush=True)
        R = g.rref(B)
        ctx.synchronize()
    finally:
        assert all([runtime.hipFree(x) == 0 for x in ballast if x.value])
    assert np.array_equal(g.Array(R), expect)
