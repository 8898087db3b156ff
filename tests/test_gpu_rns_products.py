"""Which side of the bound on the rows' sums a multi-modular product takes: one int8
product fewer where the largest sum meets it, all of them where it does not, where the
worst case is below it anyway, and with one plane."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

QLIST = [256, 255, 253, 251, 247, 241, 239, 233, 229, 227, 223, 211]


def moduli(p, k):
    """Planes of a product k deep, the product of all moduli but the last, floor(p/2)."""
    h, M = p // 2, 1
    for j, q in enumerate(QLIST):
        if M * q > 4 * k * h * h:
            return j + 1, M, h
        M *= q
    raise AssertionError


@pytest.mark.parametrize("p,k", [(2 ** 26 - 5, 8192), (2 ** 26 - 5, 5000), (2 ** 26 - 5, 1000), (65521, 1500), (8388593, 900),
                                 (1021, 12000), (127, 500)])
def test_sides(gffm, p, k):
    g, ctx = gffm, gffm.Context()
    m, n = 200, 70
    assert ctx.rns_products() == (0, 0)
    r, M, h = (1, 1, p // 2) if p <= 255 else moduli(p, k)
    asked = p > 255 and M > k * h * h + k * h * h // 32
    # the rows' sums are taken in eights, rounded up in pieces of 16
    limit = 0.498 * M / h
    rows = {"uniform": np.random.default_rng(k).integers(0, p, (m, k)), "largest": np.full((m, k), h),
            "none": np.zeros((m, k), dtype=np.int64)}
    v = int(limit / (k + 8)) - 8
    if asked and 0 < v < h - 64:
        rows["below"] = np.full((m, k), v)
        rows["above"] = np.full((m, k), min(h, int(limit / k) + 1))
        rows["one above"] = rows["none"].copy()
        rows["one above"][177] = min(h, int(limit / k) + 1)
    sides = set()
    for name, A in rows.items():
        B = np.random.default_rng(k + 1).integers(0, p, (k, n))
        balanced = np.where(A > h, A - p, A)
        pieces = np.pad(np.abs(balanced), ((0, 0), (0, -k % 16))).reshape(m, -1, 16).sum(2)
        top = 8 * int((-(-pieces // 8)).sum(1).max())
        fewer = asked and top * h < 0.498 * M
        sides.add(fewer)
        print(f"p={p} k={k} planes={r} {name}: one fewer {fewer}", flush=True)
        Ag, Bg = g.CuModMatrix(A, p, elem_type=np.float64, ctx=ctx), g.CuModMatrix(B, p, elem_type=np.float64, ctx=ctx)
        C = g.zeros(np.float64, m, n, p, ctx=ctx)
        g.mul_(C, Ag, Bg, form=3)
        assert ctx.rns_products() == (r - int(fewer), r), name
        assert np.array_equal(g.Array(C).astype(np.int64), O.gemm(A, B, p)), name
    assert len(sides) == (2 if "below" in rows else 1)
