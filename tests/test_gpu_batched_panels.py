"""Batched products through the row-panel items (k <= 256) at every remainder of
their 32-deep stages and of their 64-wide tiles, bit-exact against the oracle, with
entries that are residues and entries that are not."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

KS = list(range(0, 70)) + [95, 96, 97, 127, 128, 129, 255, 256]


@pytest.mark.parametrize("et", [np.float64, np.float32])
@pytest.mark.parametrize("p", [2, 251, 65521, 2 ** 23 - 15, 2 ** 26 - 5])
def test_row_panel_remainders(gffm, p, et):
    if et == np.float32 and p > 2 ** 12:
        pytest.skip("storage limit")
    g = gffm
    print(f"row panels p={p} {np.dtype(et).name}", flush=True)
    jobs, want = [], []
    for i, k in enumerate(KS):
        m, n = (1, 63, 64, 65, 130)[i % 5], (64, 1, 200, 33, 127, 65)[i % 6]
        Ah = O.draw_matrix(m, k, p, seed=i) if k else np.zeros((m, 0), dtype=np.int64)
        Bh = O.draw_matrix(k, n, p, seed=i, offset=m * k) if k else np.zeros((0, n), dtype=np.int64)
        Ah[:, : k // 2] = p - 1
        A, B = g.CuModMatrix(Ah, p, elem_type=et), g.CuModMatrix(Bh, p, elem_type=et)
        if i % 3 == 0 and k:
            # raw storage: the constructors reduce
            for X, H, s in ((A, Ah, -p), (B, Bh, p)):
                host = np.zeros(X.data.nbytes // np.dtype(et).itemsize, dtype=et)
                X.data.download(host)
                host.reshape(-1, X.ld)[: H.shape[1], : H.shape[0]] = (H + s * (np.arange(H.size).reshape(H.shape) % 2)).T
                X.data.upload(host)
        jobs.append((A, B, g.zeros(et, m, n, p), p))
        want.append(O.gemm(Ah, Bh, p) if k else np.zeros((m, n), dtype=np.int64))
    g.gemm_batched(jobs, et)
    g.context().synchronize()
    for (_, _, C, _), W, k in zip(jobs, want, KS):
        assert np.array_equal(g.Array(C).astype(np.int64), W), f"k={k}"
