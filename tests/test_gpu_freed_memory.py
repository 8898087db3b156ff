"""Device memory that comes back from modp_free and is handed out again: sizes
on either side of what a block may serve, freed twice, more than what is kept,
and a view of it that another stream still reads when it is freed."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KEPT = 1 << 30


def alloc(ctx, nbytes):
    p = ctypes.c_void_p()
    assert ctx.lib.modp_malloc(ctx.h, nbytes, ctypes.byref(p)) == 0
    return p


@pytest.mark.parametrize("nbytes", [1, 4096, 8 * 1000003, 64 << 20])
def test_reuse(gffm, nbytes):
    ctx = gffm.context()
    first = alloc(ctx, nbytes)
    other = alloc(ctx, nbytes)
    assert first.value != other.value
    assert ctx.lib.modp_free(ctx.h, first) == 0
    assert ctx.lib.modp_free(ctx.h, first) != 0  # twice
    larger = alloc(ctx, 2 * nbytes + 8)  # the block is too small for this
    assert larger.value != first.value
    again = alloc(ctx, nbytes)
    assert again.value not in (other.value, larger.value)
    for p in (other, larger, again):
        assert ctx.lib.modp_free(ctx.h, p) == 0


def free_bytes():
    with open("/proc/self/maps") as maps:  # the HIP runtime that the library uses
        path = next(line.split()[-1] for line in maps if "libamdhip64" in line)
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert ctypes.CDLL(path).hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_bounded(gffm):
    ctx = gffm.context()
    gffm.zeros(np.float64, 64, 64, 11)
    before = free_bytes()
    blocks = [alloc(ctx, (300 + i) << 20) for i in range(8)]
    for p in blocks:
        assert ctx.lib.modp_free(ctx.h, p) == 0
    huge = alloc(ctx, 2 * KEPT)
    assert ctx.lib.modp_free(ctx.h, huge) == 0
    assert free_bytes() >= before - KEPT - (64 << 20)


def test_read_on_another_stream(gffm):
    # a context of its own, and so another stream, reads what the first frees
    n, p = 2500, 2 ** 26 - 5
    other = gffm.Context()
    A = gffm.rand(np.float64, n, n, p, seed=4)
    expect = gffm.Array(A * A)
    for _ in range(3):
        B = gffm.rand(np.float64, n, n, p, seed=4)
        C = gffm.zeros(np.float64, n, n, p, ctx=other)
        gffm.context().synchronize()
        other.synchronize()
        for _ in range(4):
            other.check(other.lib.modp_gemm(other.h, 0, B.dtype_code, n, n, n, B.ptr, B.ld,
                                            B.ptr, B.ld, C.ptr, C.ld, p), "gemm")
        del B  # freed while the products are still to run
        D = gffm.rand(np.float64, n, n, p, seed=5)
        other.synchronize()
        assert np.array_equal(gffm.Array(C), expect)
        del D
