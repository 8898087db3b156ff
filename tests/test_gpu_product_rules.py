"""What the automatic choice takes where a form or a tile stops being the faster one,
and the products there, bit-exact against the oracle."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

PLAIN, DIGITS = 1, 2
P = {1: 127, 2: 65521, 3: 2 ** 23 - 15, 4: 2 ** 26 - 5}  # by digits


def check(g, m, n, k, p):
    Ah, Bh = O.draw_matrix(m, k, p, 51), O.draw_matrix(k, n, p, 52)
    A, B = g.CuModMatrix(Ah, p, elem_type=np.float64), g.CuModMatrix(Bh, p, elem_type=np.float64)
    C = g.zeros(np.float64, m, n, p)
    g.mul_(C, A, B)
    assert np.array_equal(g.Array(C).astype(np.int64), O.gemm(Ah, Bh, p))


# narrow products keep 64 x 64 tiles
@pytest.mark.parametrize("m,n,k,digits,tile", [
    (40000, 16, 300, 1, 64), (64, 40000, 300, 1, 64), (65, 40000, 300, 1, 128), (40000, 192, 300, 1, 128),
    (40000, 64, 300, 2, 64), (40000, 65, 300, 2, 128), (192, 20000, 300, 2, 64), (12000, 320, 300, 2, 64),
    (12000, 420, 300, 2, 128), (2501, 1203, 300, 2, 128), (2048, 2048, 300, 2, 128)])
def test_narrow_tiles(gffm, m, n, k, digits, tile):
    g, p = gffm, P[digits]
    print(f"tiles {m}x{n}x{k} p={p}", flush=True)
    cfg, _ = g.context().gemm_config(m, n, k, p)
    assert cfg["form"] == DIGITS and cfg["tile_m"] == cfg["tile_n"] == tile
    check(g, m, n, k, p)


# shallow products take the plain form: below 1000 x 1000, where they are long and thin,
# and elsewhere
@pytest.mark.parametrize("m,n,starts", [
    (64, 6000, (56, 64, 88, 96)), (1000, 1000, (56, 64, 88, 96)), (1024, 1025, (48, 48, 56, 96)),
    (40000, 8, (48, 56, 112, 112)), (64, 16400, (48, 56, 112, 112)), (100000, 16, (48, 48, 56, 96)),
    (65, 40000, (48, 48, 56, 96)), (2000, 2000, (48, 48, 56, 96))])
def test_digits_from(gffm, m, n, starts):
    g = gffm
    for digits, k in zip(P, starts):
        p = P[digits]
        print(f"digits from {m}x{n}x{k} p={p}", flush=True)
        for kk, form in ((k - 1, PLAIN), (k, DIGITS)):
            cfg, _ = g.context().gemm_config(m, n, kk, p)
            assert cfg["form"] == form, (p, kk)
            check(g, m, n, kk, p)


# the small plain kernel, and 64 x 64 tiles of one or two stages of K
@pytest.mark.parametrize("p", [11, 65521, 2 ** 26 - 5])
@pytest.mark.parametrize("m,n,k,small", [
    (17, 17, 16, False), (512, 512, 16, False), (512, 512, 17, True), (64, 64, 32, False), (64, 64, 33, True),
    (65, 64, 32, True), (65, 64, 16, False), (1, 3, 1, False), (513, 512, 40, False)])
def test_small_plain_from(gffm, m, n, k, small, p):
    g = gffm
    ctx = g.context()
    print(f"small plain {m}x{n}x{k} p={p}", flush=True)
    ctx.kernel_timing_reset()
    ctx.kernel_timing(True)
    try:
        check(g, m, n, k, p)
        assert ctx.kernel_time("gemm_f64")[1] == 1
        assert ctx.kernel_time("gemm_f64_small")[1] == int(small)
    finally:
        ctx.kernel_timing(False)
        ctx.kernel_timing_reset()
