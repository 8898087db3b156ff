"""Freed device memory that the contexts of a device share: one table of what is
kept, a block that several threads free at once, many small ones, one whose
address came back after something else had released it, and giving it all back."""
import ctypes
import threading

import pytest

pytestmark = pytest.mark.gpu


def alloc(ctx, nbytes):
    p = ctypes.c_void_p()
    assert ctx.lib.modp_malloc(ctx.h, nbytes, ctypes.byref(p)) == 0
    return p


def free(ctx, p):
    return ctx.lib.modp_free(ctx.h, p)


def hip():
    with open("/proc/self/maps") as maps:  # the HIP runtime that the library uses
        return ctypes.CDLL(next(line.split()[-1] for line in maps if "libamdhip64" in line))


def allocated(runtime, p):
    """Bytes of the runtime's allocation at p, 0 if there is none."""
    base, size = ctypes.c_void_p(), ctypes.c_size_t()
    if runtime.hipMemGetAddressRange(ctypes.byref(base), ctypes.byref(size), p) != 0:
        runtime.hipGetLastError()
        return 0
    return size.value


@pytest.mark.parametrize("nbytes", [12345, 33 << 20])
def test_contexts_share_what_is_freed(gffm, nbytes):
    one, two = gffm.context(), gffm.Context()
    p = alloc(one, nbytes)
    assert free(two, p) == 0
    assert free(one, p) != 0 and free(two, p) != 0  # freed already
    q = alloc(two, nbytes)
    assert q.value == p.value
    r = alloc(one, nbytes)
    assert r.value != q.value
    assert free(one, q) == 0 and free(two, r) == 0


def test_reused_at_once(gffm):
    # the same block again, also for up to an eighth less, not for more or much less
    ctx, n = gffm.context(), 7777777
    p = alloc(ctx, n)
    assert free(ctx, p) == 0
    for size, same in ((n, True), (n - n // 10, True), (n // 2, False), (n + 4096, False)):
        q = alloc(ctx, size)
        assert (q.value == p.value) == same, size
        assert free(ctx, q) == 0


def test_freed_by_several_threads_at_once(gffm):
    # one of them frees it, the others are told so, and it is handed out once
    contexts = [gffm.Context() for _ in range(4)]
    n = 1234567
    for _ in range(50):
        p, status = alloc(contexts[0], n), []
        start = threading.Barrier(len(contexts))

        def work(ctx):
            start.wait()
            status.append(free(ctx, p))

        threads = [threading.Thread(target=work, args=(c,)) for c in contexts]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert sorted(s == 0 for s in status) == [False, False, False, True]
        q, r = alloc(contexts[1], n), alloc(contexts[2], n)
        assert q.value != r.value
        assert free(contexts[1], q) == 0 and free(contexts[2], r) == 0


@pytest.mark.parametrize("nbytes", [1, 5000])
def test_small_blocks_are_bounded(gffm, nbytes):
    # as many as there are large pages in 1 GiB, the latest ones
    ctx, runtime = gffm.context(), hip()
    blocks = [alloc(ctx, nbytes + i) for i in range(1500)]
    assert all(allocated(runtime, p) for p in blocks)
    for p in blocks:
        assert free(ctx, p) == 0
    left = [p for p in blocks if allocated(runtime, p)]
    assert len(left) <= 512 and left[-1].value == blocks[-1].value


@pytest.mark.parametrize("n", [48 << 20, 1 << 20, 100000])
def test_address_that_came_back(gffm, n):
    ctx, runtime = gffm.context(), hip()
    runtime.hipMalloc.argtypes = [ctypes.c_void_p, ctypes.c_size_t]
    for size in (n - 1, n - 4096, n - 70000):
        p = alloc(ctx, n)
        assert allocated(runtime, p) >= n
        assert runtime.hipFree(p) == 0
        q = ctypes.c_void_p()
        assert runtime.hipMalloc(ctypes.byref(q), size) == 0
        print(n, size, hex(p.value), hex(q.value), flush=True)
        assert free(ctx, q) == 0
        r = alloc(ctx, n)
        assert allocated(runtime, r) >= n
        assert free(ctx, r) == 0
        again = alloc(ctx, n)
        assert again.value == r.value
        assert runtime.hipFree(again) == 0


def test_release(gffm):
    ctx, other, runtime = gffm.context(), gffm.Context(), hip()
    ctx.release_freed()
    assert ctx.release_freed() == 0
    blocks = [alloc(ctx, n) for n in (1, 100000, 300 << 20)]
    for p in blocks:
        assert free(ctx, p) == 0
    assert other.release_freed() >= (300 << 20) + 100001
    assert not any(allocated(runtime, p) for p in blocks)
    assert ctx.release_freed() == 0
    assert ctx.lib.modp_release_freed(ctx.h, None) == 0


def test_freed_after_the_context(gffm):
    lib, runtime = gffm.context().lib, hip()
    h, p = ctypes.c_void_p(), ctypes.c_void_p()
    assert lib.modp_ctx_create(0, ctypes.byref(h)) == 0
    assert lib.modp_malloc(h, 3 << 20, ctypes.byref(p)) == 0
    assert lib.modp_ctx_destroy(h) == 0
    assert allocated(runtime, p) >= 3 << 20
    assert lib.modp_free(h, p) == 0 and lib.modp_free(h, None) == 0
    assert allocated(runtime, p) == 0
    assert lib.modp_ctx_destroy(h) != 0  # once
