"""The allocation-free product at the size of its scratch: taken while the digit
planes rounded up to 64 fit in it, whatever tile a larger scratch would suit."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

SCRATCH = 64 << 20


def planes(m, n, k, L):
    return L * (-(-m // 64) + -(-n // 64)) * 64 * (-(-k // 64) * 64)


@pytest.mark.parametrize("m,n,k,p,L", [(4480, 4544, 3712, 65521, 2), (2112, 1984, 16384, 127, 1), (2047, 2049, 8000, 65521, 2)])
def test_planes_that_just_fit(gffm, m, n, k, p, L):
    g = gffm
    need = planes(m, n, k, L)
    print(f"noalloc {m}x{n}x{k} p={p}: {need} bytes", flush=True)
    A, B = g.rand(np.float64, m, k, p, seed=51), g.rand(np.float64, k, n, p, seed=52)
    C = g.zeros(np.float64, m, n, p)
    ctx = A.ctx
    assert need <= SCRATCH
    assert ctx.lib.modp_gemm_noalloc(ctx.h, 0, m, n, k, A.ptr, A.ld, B.ptr, B.ld, C.ptr, C.ld, p) == 0, \
        ctx.lib.modp_last_error(ctx.h)
    rows = [0, 1, 63, 64, m // 2, m - 65, m - 1]
    got = g.Array(C).astype(np.int64)
    assert np.array_equal(got[rows], O.gemm(np.ascontiguousarray(g.Array(A).astype(np.int64)[rows]),
                                            g.Array(B).astype(np.int64), p))
    D = g.zeros(np.float64, m, n, p)
    g.mul_(D, A, B, form=g.FORM_PLAIN_F64)
    assert np.array_equal(got, g.Array(D).astype(np.int64))


def test_planes_that_do_not_fit(gffm):
    g, m, n, k, p = gffm, 2176, 1984, 16384, 127
    assert planes(m, n, k, 1) > SCRATCH
    A, B, C = g.zeros(np.float64, m, k, p), g.zeros(np.float64, k, n, p), g.zeros(np.float64, m, n, p)
    ctx = A.ctx
    assert ctx.lib.modp_gemm_noalloc(ctx.h, 0, m, n, k, A.ptr, A.ld, B.ptr, B.ld, C.ptr, C.ld, p) == 8
