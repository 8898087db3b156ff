"""Triangular inverses at the edges of the 16, 32 and 64-row steps inside a diagonal
block and of the levels above it (a last pair of any size), against T X = I and the
zero triangle."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p", [2, 65521, 2 ** 24 - 3, 2 ** 26 - 5])
@pytest.mark.parametrize("upper", [True, False], ids=["upper", "lower"])
def test_triangular_sizes(gffm, upper, p):
    g = gffm
    f = g.upper_triangular_inverse_no_copy if upper else g.lower_triangular_inverse_no_copy
    tri = np.triu if upper else np.tril
    for n in (1, 15, 16, 17, 31, 32, 33, 48, 63, 65, 127, 128, 129, 191, 192, 193, 256, 257, 320, 385, 511, 513, 700, 1025):
        print(f"triangular inverse n={n} upper={upper} p={p}", flush=True)
        rng = np.random.default_rng(n)
        T = tri(rng.integers(0, p, (n, n)))
        T[np.arange(n), np.arange(n)] = rng.integers(1, p, n)
        X = g.Array(f(g.CuModMatrix(T, p, elem_type=np.float64))).astype(np.int64)
        assert np.array_equal(X, tri(X)) and X.min() >= 0 and X.max() < p
        assert np.array_equal(O.gemm(T, X, p), np.eye(n, dtype=np.int64))
