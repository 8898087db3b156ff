"""Eliminations whose panels find no pivot among the first 64 rows, or no pivot at all:
how many panels they launch, and the results against the oracle."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

KERNELS = ("one", "xcd", "global", "any")


def launches(ctx, run):
    ctx.kernel_timing_reset()
    ctx.kernel_timing(True)
    try:
        out = run()
    finally:
        ctx.kernel_timing(False)
    return {k: ctx.kernel_time("elim_panel_" + k)[1] for k in KERNELS}, out


def matrix(name, m, n, p):
    A = O.draw_matrix(m, n, p, seed=m + n)
    if name == "zero columns":
        A[:, ::3] = 0
    elif name == "sparse":
        A = np.where(O.draw_matrix(m, n, 1000, seed=7) < 1000 // n + 1, A, 0)
    elif name == "rank 1":
        A = np.ones((m, n), dtype=np.int64)
    elif name == "zero":
        A = np.zeros((m, n), dtype=np.int64)
    elif name == "rows below":
        A[:64] = 0
    elif name == "equal columns":
        A[:, 40] = A[:, 39]
    return A


NAMES = ["zero columns", "sparse", "rank 1", "zero", "rows below", "equal columns"]


@pytest.mark.parametrize("p", [7, 65521, 2 ** 26 - 5])
@pytest.mark.parametrize("name", NAMES)
def test_one_block(gffm, name, p):
    # at most one panel of any pivots per 32 columns, and the block once more
    g, n = gffm, 100
    Ah = matrix(name, n, n, p)
    A = g.CuModMatrix(Ah, p, elem_type=np.float64)
    count, R = launches(A.ctx, lambda: g.rref(A))
    print(name, p, count, flush=True)
    assert count["any"] == 4 and count["one"] <= 4
    assert np.array_equal(g.Array(R).astype(np.int64), O.rref(Ah, p)["R"])
    count, (ok, _) = launches(A.ctx, lambda: g.is_invertible_with_inverse(A))
    assert ok == (O.rref(Ah, p)["rank"] == n)
    assert count["any"] == 4 and count["one"] <= 4
    count, _ = launches(A.ctx, lambda: g.lu_full(A))
    assert count["any"] == 0 and count["one"] == 4


@pytest.mark.parametrize("p", [7, 65521, 2 ** 26 - 5])
@pytest.mark.parametrize("m,n", [(300, 300), (700, 520), (90, 400), (400, 90), (1100, 1100)])
@pytest.mark.parametrize("name", NAMES)
def test_stops(gffm, name, m, n, p):
    g = gffm
    print(name, m, n, p, flush=True)
    Ah = matrix(name, m, n, p)
    A = g.CuModMatrix(Ah, p, elem_type=np.float64)
    ref = O.rref(Ah, p)
    R, pivots, rank = g.rref_full(A)
    assert rank == ref["rank"] and np.array_equal(g.Array(R).astype(np.int64), ref["R"])
    if m == n:
        ok, X = g.is_invertible_with_inverse(A)
        assert ok == (rank == n)
        if ok:
            assert np.array_equal(O.gemm(Ah, g.Array(X).astype(np.int64), p), np.eye(n, dtype=np.int64))
    U, L, perm, piv, rank = g.lu_full(A)
    ref = O.lu(Ah, p)
    assert rank == ref["rank"] and perm == ref["perm"].tolist() and piv == ref["pivcols"].tolist()
    assert np.array_equal(g.Array(U).astype(np.int64), ref["U"])
    assert np.array_equal(g.Array(L).astype(np.int64), ref["L"])
    if m * n <= 160000:
        U, L, P, Q, rank = g.pluq(A)
        ref = O.pluq(Ah, p, O.PLUQ_OPTC)
        assert rank == ref["rank"] and P == ref["row_swaps"] and Q == ref["col_swaps"]
        assert np.array_equal(g.Array(U).astype(np.int64), ref["U"])
        assert np.array_equal(g.Array(L).astype(np.int64), ref["L"])


@pytest.mark.parametrize("p", [7, 65521, 2 ** 26 - 5])
@pytest.mark.parametrize("name", ["rank 1", "zero"])
def test_blocks_after_a_stop(gffm, name, p):
    # the host sees that the first panel stopped long before it has enqueued eight blocks
    g, n = gffm, 2000
    A = g.CuModMatrix(matrix(name, n, n, p), p, elem_type=np.float64)
    for what in (g.rref, g.pluq, g.lu, g.is_invertible_with_inverse):
        # (a first call waits for its allocations, and a busy device is late)
        counts = [sum(launches(A.ctx, lambda: what(A))[0].values()) for _ in range(6)]
        print(name, p, what.__name__, counts, flush=True)
        assert min(counts) <= 24  # of 32 in a batch
