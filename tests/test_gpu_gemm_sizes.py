"""Products at the sizes where a kernel or a rule of the automatic choice
ends: the small plain kernel (16 x 16 blocks, K in four shares), the digit
form's tiles, its two recombinations, the joint split of both operands.
Bit-exact against the oracle."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def check(g, m, n, k, p, et=np.float64, unreduced=False, **how):
    Ah = O.draw_matrix(m, k, p, seed=m + k)
    Bh = O.draw_matrix(k, n, p, seed=n, offset=m * k)
    Ah[m // 2, :] = p - 1  # extreme residues on both sides
    Bh[:, n // 2] = p - 1
    Ah[0, :] = (p - 1) // 2
    Bh[:, 0] = (p + 1) // 2 % p
    ref = O.gemm(Ah, Bh, p)
    if unreduced:  # entries outside [0, p), not reduced by the constructor
        Ah = Ah - p * (np.arange(k) % 3)[None, :]
        Bh = Bh + p * (np.arange(n) % 2)[None, :]
    A, B = (g.CuModMatrix(x, p, mod=False, elem_type=et) for x in (Ah, Bh))
    C = g.zeros(et, m, n, p)
    g.mul_(C, A, B, **how)
    assert np.array_equal(g.Array(C).astype(np.int64), ref)
    pad = C.padded_array()
    assert not pad[m:].any() and not pad[:, n:].any()


@pytest.mark.parametrize("p", [2, 2887, 65521, 2 ** 26 - 5])
@pytest.mark.parametrize("m,n,k", [(1, 2, 1), (15, 17, 3), (16, 16, 16), (17, 31, 17), (33, 15, 129), (48, 40, 56),
                                   (100, 3, 1024), (512, 512, 5), (500, 512, 130), (513, 512, 128)])
def test_small_plain(gffm, m, n, k, p):
    print(f"small plain {m}x{n}x{k} p={p}", flush=True)
    check(gffm, m, n, k, p, unreduced=True, form=1)
    check(gffm, m, n, k, p)
    if p == 2887:
        check(gffm, m, n, k, p, et=np.float32, form=1)


@pytest.mark.parametrize("p", [2, 251, 257, 65521, 65537, 2 ** 24 - 3, 2 ** 24 + 43, 2 ** 26 - 5])
@pytest.mark.parametrize("tile", [(64, 64), (128, 64), (128, 128)], ids=str)
def test_digit_tiles(gffm, tile, p):
    if tile == (128, 128) and p > 65536:
        pytest.skip("two digits at most")
    how = dict(config=dict(form=2, tile_m=tile[0], tile_n=tile[1], ksplit=1))
    # whole tiles, one row and column over, and K about the 64-deep stages
    for m, n, k in [(128, 128, 64), (129, 193, 65), (127, 63, 191), (256, 130, 256), (1, 300, 130)]:
        print(f"digit tile={tile} {m}x{n}x{k} p={p}", flush=True)
        check(gffm, m, n, k, p, unreduced=True, **how)


@pytest.mark.parametrize("p,k", [(2 ** 23 - 15, 2047), (2 ** 23 - 15, 6000), (2 ** 18 - 5, 32000), (65521, 40000),
                                 (2 ** 26 - 5, 33000)])
def test_digit_recombination(gffm, p, k):
    # on both sides of the bound up to which the digit sums are not reduced
    # first, and over more than one int32-safe piece of K
    print(f"digit recombination k={k} p={p}", flush=True)
    check(gffm, 70, 66, k, p, form=2)


@pytest.mark.parametrize("m,n,k", [(2817, 3000, 1600), (3073, 2818, 1536)])
def test_one_digit_wide_tiles(gffm, m, n, k):
    print(f"wide tiles {m}x{n}x{k}", flush=True)
    check(gffm, m, n, k, 11, et=np.float32)
    check(gffm, m, n, k, 251, form=2)


@pytest.mark.parametrize("m,n,k", [(40, 40, 5000), (300, 200, 2048), (700, 600, 4097)])
@pytest.mark.parametrize("p", [11, 65521, 2 ** 23 - 15, 2 ** 26 - 5])
def test_automatic_k_slices(gffm, m, n, k, p):
    print(f"k slices {m}x{n}x{k} p={p}", flush=True)
    check(gffm, m, n, k, p)
