"""The multi-modular form with one modulus fewer than the worst case asks for: taken
when the rows' sums allow it, refused otherwise, bit-exact against the oracle on both
sides of the bound (the largest sums that meet it, and the smallest that do not)."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

QLIST = [256, 255, 253, 251, 247, 241, 239, 233, 229, 227, 223, 211]


def moduli(p, k):
    h, M = p // 2, 1
    for j, q in enumerate(QLIST):
        if M * q > 4 * k * h * h:
            return j + 1, M, h
        M *= q
    raise AssertionError


CASES = [(2 ** 26 - 5, 8192), (2 ** 26 - 5, 5000), (65521, 1500), (8388593, 900), (2 ** 24 - 3, 33), (1021, 12000)]


@pytest.mark.parametrize("p,k", CASES)
def test_bound_sides(gffm, p, k):
    g = gffm
    r, M, h = moduli(p, k)
    assert M > 1
    inside = M > k * h * h + k * h * h // 32  # else always all moduli
    m, n = 131, 70
    rng = np.random.default_rng(k)
    sign = lambda s: np.where(rng.random(s) < 0.5, -1, 1)
    full = np.full((m, k), h, dtype=np.int64)
    c = min(h, max(1, int(0.498 * M / (h * k)) - 8))
    cases = {"random": (rng.integers(0, p, (m, k)), rng.integers(0, p, (k, n))),
             "worst": (full, np.full((k, n), h, dtype=np.int64)),
             "worst mixed": (full * sign((m, k)), h * sign((k, n)))}
    for name, v in (("below", c), ("above", min(h, c + 64))):
        cases[name] = (np.full((m, k), v), np.full((k, n), -h))
        A = np.zeros((m, k), dtype=np.int64)
        A[77] = v
        cases[name + ", one row"] = (A, h * sign((k, n)))
    for name, (A, B) in cases.items():
        print(f"p={p} k={k} r={r} inside={inside} {name}", flush=True)
        A, B = A % p, B % p
        C = g.zeros(np.float64, m, n, p)
        Ag, Bg = g.CuModMatrix(A, p, elem_type=np.float64), g.CuModMatrix(B, p, elem_type=np.float64)
        for _ in range(2):  # the sums start again from zero
            g.mul_(C, Ag, Bg, form=3)
            assert np.array_equal(g.Array(C).astype(np.int64), O.gemm(A, B, p)), name
