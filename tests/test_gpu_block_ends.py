"""Updates inside an outer block and its end (rows of U by the panels' inverse
triangles, composed row moves) where tiles, panels and blocks are ragged, bit-exact
against the oracle: one to sixteen columns beside a block, blocks of fewer than
128 pivots, pivots that skip columns, 16-column panels, and moduli on both sides
of the one-reduction bound and of the table of inverses."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def draw(m, n, rank, p, seed):
    if rank >= min(m, n):
        return O.draw_matrix(m, n, p, seed)
    return O.gemm(O.draw_matrix(m, rank, p, seed), O.draw_matrix(rank, n, p, seed, offset=m * rank), p)


CASES = [
    # m, n, rank, columns set to zero
    (33, 49, 33, ()), (129, 129, 129, ()), (130, 145, 130, ()), (300, 161, 161, ()), (161, 305, 150, ()),
    (290, 290, 290, (5, 40, 41, 129, 200)), (400, 270, 140, (0, 127, 128)),
]


@pytest.mark.parametrize("wide", [False, True], ids=["panel32", "panel16"])
@pytest.mark.parametrize("p", [2, 65521, 131071, 262147, 2 ** 24 - 3, 2 ** 26 - 5])
@pytest.mark.parametrize("m,n,rank,zero", CASES)
def test_block_ends_vs_oracle(gffm, monkeypatch, m, n, rank, zero, p, wide):
    if wide:
        monkeypatch.setenv("MODP_PANEL_GLOBAL", "1")
    print(f"block ends m={m} n={n} rank={rank} zero={zero} p={p} wide={wide}", flush=True)
    Ah = draw(m, n, rank, p, seed=7 * m + n)
    Ah[:, list(zero)] = 0

    def dev():
        return gffm.CuModMatrix(Ah, p, elem_type=np.float64)

    U, L, P, Q, r = gffm.pluq(dev(), form=0)
    ref = O.pluq(Ah, p, O.PLUQ_OPTC)
    assert r == ref["rank"] and P == ref["row_swaps"] and Q == ref["col_swaps"]
    assert np.array_equal(gffm.Array(U).astype(np.int64), ref["U"])
    assert np.array_equal(gffm.Array(L).astype(np.int64), ref["L"])
    U, L, perm, piv, r = gffm.lu_full(dev())
    ref = O.lu(Ah, p)
    assert r == ref["rank"] and perm == ref["perm"].tolist() and piv == ref["pivcols"].tolist()
    assert np.array_equal(gffm.Array(U).astype(np.int64), ref["U"])
    assert np.array_equal(gffm.Array(L).astype(np.int64), ref["L"])
    R, piv, r = gffm.rref_full(dev())
    ref = O.rref(Ah, p)
    assert r == ref["rank"] and piv == ref["pivcols"].tolist()
    assert np.array_equal(gffm.Array(R).astype(np.int64), ref["R"])
