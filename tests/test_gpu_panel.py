"""The register panel of the eliminations at the sizes where it can go wrong:
one workgroup against several (256 rows), partly filled waves, panels narrower
than 32 columns, more slots than lanes (over 4096 rows), the three arithmetic
modes and the two rounds of its pivot inverse at the boundaries of the modulus,
zero columns inside a panel, moduli that are not prime, and panels whose
workgroups give up waiting for each other.  Bit-exact against the oracle."""
from math import gcd

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def all_modes_equal(g, Ah, p):
    A = g.CuModMatrix(Ah, p, elem_type=np.float64)
    U, L, P, Q, rank = g.pluq(A)
    ref = O.pluq(Ah, p, O.PLUQ_OPTC)
    assert rank == ref["rank"] and P == ref["row_swaps"] and Q == ref["col_swaps"]
    assert np.array_equal(g.Array(U).astype(np.int64), ref["U"])
    assert np.array_equal(g.Array(L).astype(np.int64), ref["L"])
    U, L, perm, piv, rank = g.lu_full(A)
    ref = O.lu(Ah, p)
    assert rank == ref["rank"] and perm == ref["perm"].tolist() and piv == ref["pivcols"].tolist()
    assert np.array_equal(g.Array(U).astype(np.int64), ref["U"])
    assert np.array_equal(g.Array(L).astype(np.int64), ref["L"])


# 1021 and 1031 lie on either side of the table of inverses, 65521 and 65537 of
# the 16-bit keys, 2^24 - 3 and 2^24 + 43 of the reduced updates, 2^18 - 5 and
# 2^18 + 3 of the inverse's second round
PRIMES = [2, 3, 1021, 1031, 65521, 65537, 2 ** 18 - 5, 2 ** 18 + 3, 2 ** 24 - 3, 2 ** 24 + 43, 2 ** 26 - 5]


@pytest.mark.parametrize("p", PRIMES)
@pytest.mark.parametrize("shape", [(255, 40), (256, 33), (257, 32), (258, 31), (321, 65), (40, 300), (513, 130)], ids=str)
def test_panel_vs_oracle(gffm, shape, p):
    m, n = shape
    print(f"panel shape={shape} p={p}", flush=True)
    Ah = O.draw_matrix(m, n, p, seed=5)
    all_modes_equal(gffm, Ah, p)
    # zero columns inside the panels and rows that repeat
    Ah[:, [1, 7, min(n - 1, 30)]] = 0
    Ah[m // 2:] = Ah[: m - m // 2]
    all_modes_equal(gffm, Ah, p)


@pytest.mark.parametrize("m,p", [(4095, 65521), (4097, 7), (4160, 2 ** 26 - 5), (8200, 2 ** 23 - 15), (16384, 251)])
def test_panel_many_waves(gffm, m, p):
    print(f"panel m={m} p={p}", flush=True)
    all_modes_equal(gffm, O.draw_matrix(m, 40, p, seed=6), p)


@pytest.mark.parametrize("p", [7, 65521, 2 ** 26 - 5])
def test_panel_gives_up(gffm, monkeypatch, p):
    # no workgroup waits for another: the panels go to the W-resident kernel
    monkeypatch.setenv("MODP_PANEL_PATIENCE", "-1")
    print(f"panel gives up p={p}", flush=True)
    Ah = O.draw_matrix(700, 300, p, seed=7)
    Ah[:, [2, 140, 141]] = 0
    all_modes_equal(gffm, Ah, p)


@pytest.mark.parametrize("p", [1009 * 61, 8191 * 1021, 8191 * 8179])
@pytest.mark.parametrize("m", [100, 400])
def test_panel_composite_modulus(gffm, p, m):
    # every pivot a unit (the multipliers the inverse tries need not be)
    checked = 0
    for seed in range(40):
        Ah = O.draw_matrix(m, 8, p, seed=seed)
        ref = O.pluq(Ah, p, O.PLUQ_OPTC)
        if ref["rank"] == 8 and all(gcd(int(ref["L"][k, k]), p) == 1 for k in range(8)):
            print(f"composite p={p} m={m} seed={seed}", flush=True)
            all_modes_equal(gffm, Ah, p)
            checked += 1
    assert checked >= 5
