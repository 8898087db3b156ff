"""Several threads with a context each, at once: panels that wait for each other on the
same XCD, products and vectors with their own workspaces, memory freed meanwhile.
Every result against the oracle."""
import threading

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [(300, 700, 1500), (3000, 3000, 2500), (9000, 5000, 16384)], ids=str)
def test_eliminations_beside_each_other(gffm, sizes):
    g, p, n = gffm, 65521, 260
    print(f"threads {sizes}", flush=True)
    inputs = [O.draw_matrix(m, n, p, seed=m + i) for i, m in enumerate(sizes)]
    lu = [O.lu(A, p) for A in inputs]
    rref = [O.rref(A, p) for A in inputs]
    x = [O.draw_matrix(n, 1, p, seed=3 + i) for i in range(len(sizes))]
    Ax = [O.gemm(A, v, p) for A, v in zip(inputs, x)]
    failed, start = [], threading.Barrier(len(sizes))

    def work(i):
        try:
            ctx = g.Context()
            A = g.CuModMatrix(inputs[i], p, elem_type=np.float64, ctx=ctx)
            v = g.CuModMatrix(x[i], p, elem_type=np.float64, ctx=ctx)
            start.wait()
            for _ in range(3):
                U, L, perm, piv, rank = g.lu_full(A)
                assert rank == lu[i]["rank"] and perm == lu[i]["perm"].tolist(), "lu"
                assert np.array_equal(g.Array(U).astype(np.int64), lu[i]["U"]), "U"
                R, _, _ = g.rref_full(A)
                assert np.array_equal(g.Array(R).astype(np.int64), rref[i]["R"]), "rref"
                assert np.array_equal(g.Array(A * v).astype(np.int64), Ax[i]), "A x"
        except BaseException as e:  # noqa: BLE001 (reported by the test)
            failed.append((sizes[i], repr(e)))
            start.abort()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(sizes))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert failed == []
