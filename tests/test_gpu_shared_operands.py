"""Results that lie in an operand's own memory, bit-exact against the oracle of the
operands as they were: a matrix-vector product into a column of its matrix."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("et,p", [(np.float64, 65521), (np.float64, 2 ** 26 - 5), (np.float32, 2039)])
@pytest.mark.parametrize("m,k,col", [(40, 30, 29), (700, 600, 0), (3001, 2003, 1000), (6001, 7003, 7002)])
def test_gemv_into_its_matrix(gffm, m, k, col, et, p):
    g = gffm
    print(f"gemv into column {col} of {m}x{k} p={p}", flush=True)
    A, x = O.draw_matrix(m, k, p, 21), O.draw_matrix(k, 1, p, 22)
    ref = O.gemm(A, x, p)
    for _ in range(3):
        Ag = g.CuModMatrix(A, p, elem_type=et)
        xg = g.CuModVector(x[:, 0], p, elem_type=et)
        ctx = Ag.ctx
        y = Ag.ptr + Ag.elem_type.itemsize * Ag.ld * col
        ctx.check(ctx.lib.modp_gemv(ctx.h, Ag.dtype_code, m, k, Ag.ptr, Ag.ld, xg.ptr, y, p), "gemv")
        got = g.Array(Ag).astype(np.int64)
        assert np.array_equal(got[:, col:col + 1], ref)
        got[:, col] = A[:, col]
        assert np.array_equal(got, A)
