"""Matrix-vector products at the edges of their row blocks, batches and K slices,
bit-exact against the oracle: odd row counts, one to many slices, entries that are
not residues, a result that replaces the operand, and calls in a row (the slices'
counts are left at zero)."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def draw(m, k, p, seed, unreduced):
    A = O.draw_matrix(m, k, p, seed)
    x = O.draw_matrix(k, 1, p, seed + 1)
    A[0, :] = p - 1
    x[: k // 2 + 1] = p - 1
    if unreduced:
        return A, x, A - p * (np.arange(m)[:, None] % 3), x + p * (np.arange(k)[:, None] % 2)
    return A, x, A, x


@pytest.mark.parametrize("p", [2, 2039, 65521, 2 ** 26 - 5, 2 ** 26])
@pytest.mark.parametrize("m", [1, 2, 3, 5, 127, 128, 129, 255, 259, 1025])
def test_gemv_edges(gffm, m, p):
    g = gffm
    kinds = [np.float64] + ([np.float32] if p == 2039 else [])
    for k in (1, 7, 8, 33, 63, 65, 130, 577, 4099):
        print(f"gemv {m}x{k} p={p}", flush=True)
        A, x, Ad, xd = draw(m, k, p, 5 * m + k, False)
        ref = O.gemm(A, x, p)
        for et in kinds:
            Ag, xg = g.CuModMatrix(Ad, p, elem_type=et), g.CuModVector(xd[:, 0], p, elem_type=et)
            for _ in range(3):
                z = g.zeros(et, m, 1, p)
                g.mul_(z, Ag, xg)
                assert np.array_equal(g.Array(z).astype(np.int64), ref)


@pytest.mark.parametrize("m,k", [(100, 60), (129, 4099), (2, 700)])
def test_gemv_unreduced_entries(gffm, m, k):
    g, p = gffm, 65521
    A, x, Ad, xd = draw(m, k, p, 3, True)
    Ag = g.CuModMatrix(A, p, elem_type=np.float64)
    xg = g.CuModVector(x[:, 0], p, elem_type=np.float64)
    # raw storage: the constructors reduce
    host = np.zeros(Ag.data.nbytes // 8)
    Ag.data.download(host)
    host.reshape(-1, Ag.ld)[:k, :m] = Ad.T
    Ag.data.upload(host)
    host = np.zeros(xg.data.nbytes // 8)
    xg.data.download(host)
    host[:k] = xd[:, 0]
    xg.data.upload(host)
    z = g.zeros(np.float64, m, 1, p)
    g.mul_(z, Ag, xg)
    assert np.array_equal(g.Array(z).astype(np.int64), O.gemm(A, x, p))


@pytest.mark.parametrize("n", [40, 200, 1500])
def test_gemv_over_its_operand(gffm, n):
    g, p = gffm, 65521
    A, x, _, _ = draw(n, n, p, 9, False)
    Ag = g.CuModMatrix(A, p, elem_type=np.float64)
    xg = g.CuModVector(x[:, 0], p, elem_type=np.float64)
    ctx = xg.ctx
    ctx.check(ctx.lib.modp_gemv(ctx.h, 0, n, n, Ag.ptr, Ag.ld, xg.ptr, xg.ptr, p), "gemv")
    assert np.array_equal(g.Array(xg).astype(np.int64).reshape(-1, 1), O.gemm(A, x, p))
