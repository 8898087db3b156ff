"""Batched eliminations on both sides of the size from which an instance runs on
several wavefronts (more than 6144 elements, moduli below 2^16), every output
bit-exact against the oracle: edges of the tiles, zero and repeated columns, ranks
from nothing to full."""
import numpy as np
import pytest

import oracle as O
from gpufinitefieldmatrices import workloads as W

pytestmark = pytest.mark.gpu

SHAPES = [(48, 128), (49, 128), (128, 48), (128, 49), (96, 64), (97, 64), (64, 97), (80, 79), (128, 128), (127, 113),
          (100, 128), (128, 72), (66, 96)]


def instances(seed):
    rng = np.random.default_rng(seed)
    out = []
    for i, p in enumerate([2, 3, 251, 257, 65521] * 2):
        for j, (m, n) in enumerate(SHAPES):
            A = rng.integers(0, p, size=(m, n))
            kind = (i + j) % 5
            if kind == 1:    # zero columns, also first and last
                A[:, [0, 7, 8, 9, n // 2, n - 1]] = 0
            elif kind == 2:  # rank about a third
                r = min(m, n) // 3
                A = (rng.integers(0, p, (m, r)) @ rng.integers(0, p, (r, n))) % p
            elif kind == 3:  # repeated columns and zero rows
                A[:, 1::2] = A[:, : 2 * (n // 2) : 2][:, : A[:, 1::2].shape[1]]
                A[rng.choice(m, m // 3, replace=False)] = 0
            elif kind == 4 and j == 0:
                A[:] = 0
            out.append((A.astype(np.int64), p))
    return out


@pytest.mark.parametrize("op", ["pluq", "lu", "rref"])
def test_instances_on_several_waves(gffm, op):
    g = gffm
    inst = instances(21)
    arena = W.ElimArena(g.context(), inst)
    print(f"several waves {op}: {len(inst)} instances", flush=True)
    g.elim_batched({"pluq": 0, "lu": 1, "rref": 2}[op], list(arena.jobs), ctx=g.context())
    for i, (r, (A, p)) in enumerate(zip(arena.download(), inst)):
        nr, nc, rank = (int(x) for x in r["counts"])
        if op == "pluq":
            ref = O.pluq(A, p, O.PLUQ_OPTC)
            assert rank == ref["rank"], i
            assert [tuple(x) for x in r["row"][: 2 * nr].reshape(-1, 2).tolist()] == ref["row_swaps"], i
            assert [tuple(x) for x in r["col"][: 2 * nc].reshape(-1, 2).tolist()] == ref["col_swaps"], i
            assert np.array_equal(r["U"], ref["U"]) and np.array_equal(r["L"], ref["L"]), i
        elif op == "lu":
            ref = O.lu(A, p)
            assert rank == ref["rank"], i
            assert r["row"][: A.shape[0]].tolist() == ref["perm"].tolist(), i
            assert r["col"][:rank].tolist() == ref["pivcols"].tolist(), i
            assert np.array_equal(r["U"], ref["U"]) and np.array_equal(r["L"], ref["L"]), i
        else:
            ref = O.rref(A, p)
            assert rank == ref["rank"], i
            assert r["row"][:rank].tolist() == ref["pivcols"].tolist(), i
            assert np.array_equal(r["U"], ref["R"]), i
