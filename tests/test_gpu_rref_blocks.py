"""The reduced echelon form by back substitution in blocks, which a matrix takes whose
free columns leave no room for the inverse of its triangle: at the edges of the
blocks of 512 pivots and 1024 columns, and with little device memory."""
import ctypes

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def low_rank(m, n, rank, p, seed, spread):
    """rank pivots, in the first columns or all over."""
    A = O.gemm(O.draw_matrix(m, rank, p, seed), O.draw_matrix(rank, n, p, seed + 1), p)
    if spread:
        A[:, ::5] = 0
        A[:, 3::7] = A[:, 1:2]
    return A


@pytest.mark.parametrize("p,et", [(65521, np.float64), (2 ** 26 - 5, np.float64), (11, np.float32), (1009 * 61, np.float64)])
@pytest.mark.parametrize("m,n,rank,spread", [(1, 5, 1, False), (40, 60, 30, True), (513, 2000, 513, False), (700, 1537, 512, True),
                                             (600, 2500, 511, True), (1100, 1200, 1025, False), (300, 200, 120, False)])
def test_blocks(gffm, monkeypatch, m, n, rank, spread, p, et):
    g = gffm
    print(f"rref by blocks {m}x{n} rank {rank} p={p}", flush=True)
    Ah = low_rank(m, n, rank, p, 81, spread)
    if p == 1009 * 61:  # unit pivots: the identity in front
        Ah[:, :min(m, n)] = np.triu(Ah[:, :min(m, n)], 1) + np.eye(m, min(m, n), dtype=np.int64)
    A = g.CuModMatrix(Ah, p, elem_type=et)
    whole = g.Array(g.rref(A))
    monkeypatch.setenv("MODP_RREF_BLOCKS", "1")
    for form in (0, 1, 2):
        assert np.array_equal(g.Array(g.rref(A, form=form)), whole), form
    if p != 1009 * 61:
        assert np.array_equal(whole.astype(np.int64), O.rref(Ah, p)["R"])


@pytest.mark.parametrize("spread", [False, True])
def test_little_memory(gffm, spread):
    # room for the result, the elimination's own copy and 150 MB
    g, p, n, rank = gffm, 65521, 6000, 4500
    with open("/proc/self/maps") as maps:  # the HIP runtime that the library uses
        runtime = ctypes.CDLL(next(line.split()[-1] for line in maps if "libamdhip64" in line))
    runtime.hipMalloc.argtypes = [ctypes.c_void_p, ctypes.c_size_t]
    X, Y = g.rand(np.float64, n, rank, p, seed=1), g.rand(np.float64, rank, n, p, seed=2)
    A = X * Y
    if spread:
        Ah = g.Array(A)
        Ah[:, ::9] = 0
        A = g.CuModMatrix(Ah, p, elem_type=np.float64)
    expect = g.Array(g.rref(A))
    ctx = g.Context()
    B = g.CuModMatrix(g.Array(A), p, elem_type=np.float64, ctx=ctx)
    g.rref(g.rand(np.float64, 300, 300, p, seed=3, ctx=ctx))
    ctx.synchronize()
    ctx.release_freed()
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    keep = 8 * (n + 32) ** 2 + 4 * 6016 * n + (150 << 20)
    ballast = []
    try:
        for _ in range(4):  # (what is free is an estimate while much of it is)
            assert runtime.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
            if free.value <= keep + (16 << 20):
                break
            ballast.append(ctypes.c_void_p())
            assert runtime.hipMalloc(ctypes.byref(ballast[-1]), free.value - keep) == 0
        print(f"{free.value} bytes left of {total.value}", flush=True)
        R = g.rref(B)
        ctx.synchronize()
    finally:
        assert all([runtime.hipFree(x) == 0 for x in ballast if x.value])
    assert np.array_equal(g.Array(R), expect)
