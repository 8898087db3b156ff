"""Results that lie in an operand's own memory, bit-exact against the oracle of the
operands as they were: a matrix-vector product into a column of its matrix, and
products over either operand in every form."""
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


@pytest.mark.parametrize("et,p", [(np.float64, 65521), (np.float64, 2 ** 26 - 5), (np.float32, 11)])
@pytest.mark.parametrize("n", [5, 17, 48, 64, 65, 100, 200, 256, 300, 1100])
def test_product_over_an_operand(gffm, n, et, p):
    g = gffm
    A, B = O.draw_matrix(n, n, p, 31), O.draw_matrix(n, n, p, 32)
    ref = O.gemm(A, B, p)
    for form in (0, 1, 2, 3):
        print(f"n={n} p={p} form={form}", flush=True)
        for over in ("A", "B"):
            Ag, Bg = g.CuModMatrix(A, p, elem_type=et), g.CuModMatrix(B, p, elem_type=et)
            C = Ag if over == "A" else Bg
            g.mul_(C, Ag, Bg, form=form)
            assert np.array_equal(g.Array(C).astype(np.int64), ref), (form, over)


@pytest.mark.parametrize("m,k,n", [(64, 40, 300), (300, 40, 64), (200, 30, 30), (130, 130, 20)])
def test_product_into_part_of_an_operand(gffm, m, k, n):
    # C at the end of B's memory, with rows of A's stride
    g, p = gffm, 65521
    A, B = O.draw_matrix(m, k, p, 33), O.draw_matrix(k, n, p, 34)
    Ag = g.CuModMatrix(A, p, elem_type=np.float64)
    buf = np.zeros((max(m, k), 2 * n))
    buf[:k, :n] = B
    Bg = g.CuModMatrix(buf, p, elem_type=np.float64)
    ctx = Ag.ctx
    c = Bg.ptr + 8 * Bg.ld * (n // 2)
    ctx.check(ctx.lib.modp_gemm(ctx.h, 0, 0, m, n, k, Ag.ptr, Ag.ld, Bg.ptr, Bg.ld, c, Bg.ld, p), "gemm")
    assert np.array_equal(g.Array(Bg)[:m, n // 2:n // 2 + n].astype(np.int64), O.gemm(A, B, p))
