"""Which kernel factors the panels, by the rows that are left: one workgroup, the
workgroups of one XCD (all of them resident at once) or the matrix in memory.  The
launches are counted by the names of the kernel timings."""
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


@pytest.mark.parametrize("p", [251, 2 ** 23 - 15, 2 ** 26 - 5])
@pytest.mark.parametrize("m", [256, 257, 4097, 8192, 8200, 12001, 16384])
def test_panels_on_one_xcd(gffm, m, p):
    g = gffm
    Ah = O.draw_matrix(m, 150, p, seed=61)
    A = g.CuModMatrix(Ah, p, elem_type=np.float64)
    n, (U, L, P, Q, rank) = launches(A.ctx, lambda: g.pluq(A))
    print(m, p, n, flush=True)
    assert n["global"] == 0 and n["any"] == 0
    assert n["xcd"] == {256: 0, 257: 1}.get(m, 5) and n["one"] == 5 - n["xcd"]
    ref = O.pluq(Ah, p, O.PLUQ_OPTC)
    assert rank == ref["rank"] and P == ref["row_swaps"] and Q == ref["col_swaps"]
    assert np.array_equal(g.Array(U).astype(np.int64), ref["U"])
    assert np.array_equal(g.Array(L)[:, :150].astype(np.int64), ref["L"][:, :150])


def test_panels_of_more_rows(gffm):
    g, p, m = gffm, 65521, 16385
    Ah = O.draw_matrix(m, 40, p, seed=62)
    A = g.CuModMatrix(Ah, p, elem_type=np.float64)
    n, (U, L, P, Q, rank) = launches(A.ctx, lambda: g.pluq(A))
    print(m, n, flush=True)
    assert n["xcd"] == 0 and n["global"] > 0
    ref = O.pluq(Ah, p, O.PLUQ_OPTC)
    assert rank == ref["rank"] and P == ref["row_swaps"]
    assert np.array_equal(g.Array(U).astype(np.int64), ref["U"])


def test_tries_after_giving_up(gffm, monkeypatch):
    # 15 blocks, every panel on an XCD gives up: after the first batch of eight
    # blocks one block is tried at a time, with 1, 2, 4 and 8 blocks in between
    monkeypatch.setenv("MODP_PANEL_PATIENCE", "-1")
    g, p, m, blocks = gffm, 65521, 3000, 15
    Ah = O.draw_matrix(m, 128 * blocks, p, seed=63)
    A = g.CuModMatrix(Ah, p, elem_type=np.float64)
    n, (U, L, P, Q, rank) = launches(A.ctx, lambda: g.pluq(A))
    print(n, flush=True)
    assert n["one"] == 0 and n["global"] == 8 * blocks
    assert n["xcd"] == 4 * 8 + 4 * 3
    ref = O.pluq(Ah, p, O.PLUQ_OPTC)
    assert rank == ref["rank"] and P == ref["row_swaps"] and Q == ref["col_swaps"]
    assert np.array_equal(g.Array(U).astype(np.int64), ref["U"])
    assert np.array_equal(g.Array(L)[:, :rank].astype(np.int64), ref["L"][:, :rank])


def test_tries_after_giving_up_lu(gffm, monkeypatch):
    # blocks with zero columns go one by one
    monkeypatch.setenv("MODP_PANEL_PATIENCE", "-1")
    g, p, m = gffm, 65521, 1500
    Ah = O.draw_matrix(m, 128 * 7, p, seed=64)
    Ah[:, 5::100] = 0
    A = g.CuModMatrix(Ah, p, elem_type=np.float64)
    n, (U, L, perm, piv, rank) = launches(A.ctx, lambda: g.lu_full(A))
    print(n, flush=True)
    assert n["xcd"] > 0 and n["global"] > 0
    ref = O.lu(Ah, p)
    assert rank == ref["rank"] and perm == ref["perm"].tolist() and piv == ref["pivcols"].tolist()
    assert np.array_equal(g.Array(U).astype(np.int64), ref["U"])
    assert np.array_equal(g.Array(L).astype(np.int64), ref["L"])


@pytest.mark.parametrize("spins", [-1, 0, 1])
@pytest.mark.parametrize("p", [7, 65521, 2 ** 26 - 5])
@pytest.mark.parametrize("m,n", [(300, 20), (700, 300), (3000, 260)])
def test_exchange_that_does_not_end(gffm, monkeypatch, m, n, p, spins):
    # the elimination starts again from its input; from 0 on some wave may lose
    # some step, below every wave the first one
    monkeypatch.setenv("MODP_PANEL_SPINS", str(spins))
    g = gffm
    Ah = O.draw_matrix(m, n, p, seed=65)
    A = g.CuModMatrix(Ah, p, elem_type=np.float64)
    count, (U, L, P, Q, rank) = launches(A.ctx, lambda: g.pluq(A))
    print(m, n, p, spins, count, flush=True)
    assert count["xcd"] > 0 and (count["global"] > 0 or spins >= 0)
    ref = O.pluq(Ah, p, O.PLUQ_OPTC)
    assert rank == ref["rank"] and P == ref["row_swaps"] and Q == ref["col_swaps"]
    assert np.array_equal(g.Array(U).astype(np.int64), ref["U"])
    assert np.array_equal(g.Array(L).astype(np.int64), ref["L"])
    Ah[:, ::7] = 0
    A = g.CuModMatrix(Ah, p, elem_type=np.float64)
    U, L, perm, piv, rank = g.lu_full(A)
    ref = O.lu(Ah, p)
    assert rank == ref["rank"] and perm == ref["perm"].tolist() and piv == ref["pivcols"].tolist()
    assert np.array_equal(g.Array(U).astype(np.int64), ref["U"])
    assert np.array_equal(g.Array(L).astype(np.int64), ref["L"])
    # no pivot in the first rows: rref with panels that meet, too
    Ah[:64] = 0
    A = g.CuModMatrix(Ah, p, elem_type=np.float64)
    assert np.array_equal(g.Array(g.rref(A)).astype(np.int64), O.rref(Ah, p)["R"])
