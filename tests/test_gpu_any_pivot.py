"""Echelon forms and inverses whose panels take any pivot among their first 64
rows, where that can go wrong: fewer rows or columns than a panel, ragged
blocks, columns whose pivots lie further down (the general panels take over and
hand back), zero columns, singular matrices, the smallest and largest primes.
A composite modulus stays with the general panels.  Bit-exact against the
oracle."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

PRIMES = [2, 3, 251, 65521, 2 ** 18 - 5, 2 ** 18 + 3, 2 ** 24 - 3, 2 ** 24 + 43, 2 ** 26 - 5]


def shaped(m, n, p, what):
    A = O.draw_matrix(m, n, p, seed=11)
    k = min(m, n)
    if what == "zero columns":
        A[:, [0, k // 2, k - 1]] = 0
    elif what == "far pivots":  # from the middle on no pivot near the diagonal
        h = k // 2
        A[h:, h:] = 0
        A[np.arange(m - 1, m - 1 - (k - h), -1), np.arange(h, k)] = 1 + np.arange(k - h) % (p - 1)
    elif what == "far then near":  # far pivots for one stretch only
        rows = np.arange(m)
        h = min(k // 3, 40)
        A[: m // 2, h:h + 5] = 0
        A[rows >= m - 7, h:h + 5] = A[rows >= m - 7, h:h + 5] | 1
    elif what == "low rank":
        A[k // 2:] = A[: m - k // 2] if m <= 2 * (k // 2) else np.resize(A[: k // 2], (m - k // 2, n))
    return A % p


KINDS = ["random", "zero columns", "far pivots", "far then near", "low rank"]


@pytest.mark.parametrize("p", PRIMES)
@pytest.mark.parametrize("shape", [(1, 5), (5, 1), (31, 40), (33, 33), (65, 64), (100, 300), (129, 127), (300, 170), (419, 419)],
                         ids=str)
def test_rref(gffm, shape, p):
    for what in KINDS:
        print(f"rref shape={shape} p={p} {what}", flush=True)
        Ah = shaped(*shape, p, what)
        R, piv, rank = gffm.rref_full(gffm.CuModMatrix(Ah, p, elem_type=np.float64))
        ref = O.rref(Ah, p)
        assert rank == ref["rank"] and piv == ref["pivcols"].tolist()
        assert np.array_equal(gffm.Array(R).astype(np.int64), ref["R"])


@pytest.mark.parametrize("p", PRIMES)
@pytest.mark.parametrize("n", [1, 2, 31, 64, 65, 128, 193, 257, 450])
def test_inverse(gffm, n, p):
    for what in KINDS:
        print(f"inverse n={n} p={p} {what}", flush=True)
        Ah = shaped(n, n, p, what)
        ref = O.inverse(Ah, p)
        ok, X = gffm.is_invertible_with_inverse(gffm.CuModMatrix(Ah, p, elem_type=np.float64))
        assert ok == (ref is not None)
        if ok:
            assert np.array_equal(gffm.Array(X).astype(np.int64), ref)


@pytest.mark.parametrize("p", [35, 2 ** 20])
def test_composite(gffm, p):
    # a triangular matrix with units as pivots, under a modulus that has zero divisors
    Ah = np.triu(O.draw_matrix(150, 150, p, seed=3), 1) + np.eye(150, dtype=np.int64)
    X = gffm.inverse(gffm.CuModMatrix(Ah, p, elem_type=np.float64))
    assert np.array_equal(O.gemm(Ah, gffm.Array(X).astype(np.int64), p), np.eye(150, dtype=np.int64))
