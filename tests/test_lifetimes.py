"""The library's context outlives the buffers and plans that were made from it, in
whatever order Python finds them unreachable (a recording stand-in for the
library: no GPU)."""
import ctypes
import gc

import numpy as np
import pytest


class Library:
    def __init__(self):
        self.calls, self.next = [], 1

    def make(self, ref):
        ref._obj.value = self.next
        self.next += 1
        return 0

    def __getattr__(self, name):
        def call(*args):
            self.calls.append(name)
            makes = {"modp_ctx_create": 1, "modp_malloc": 2, "modp_gemm_batched_plan": 4, "modp_elim_batched_plan": 5}
            return self.make(args[makes[name]]) if name in makes else 0
        call.__name__ = name
        return call


@pytest.fixture
def library(monkeypatch):
    import gpufinitefieldmatrices as g
    lib = Library()
    monkeypatch.setattr(g._lib, "load", lambda: lib)
    return g, lib


def objects(g):
    ctx = g.Context()
    A = g.zeros(np.float64, 4, 4, 7, ctx=ctx)
    return [ctx, A, g.GemmBatchPlan([(A, A, A, 7)]), g.ElimBatchPlan(0, [], ctx=ctx), g.zeros(np.float32, 3, 2, 7, ctx=ctx)]


FREED = ["modp_ctx_destroy", "modp_elim_batched_destroy", "modp_free", "modp_free", "modp_gemm_batched_destroy"]


def released(lib):
    return [c for c in lib.calls if "destroy" in c or c == "modp_free"]


def test_in_a_cycle(library):
    g, lib = library
    for turn in range(2):
        lib.calls.clear()
        ring = objects(g)
        if turn:
            ring.reverse()
        ring.append(ring)
        gc.collect()
        assert released(lib) == []
        del ring
        gc.collect()
        assert sorted(released(lib)) == FREED and released(lib)[-1] == "modp_ctx_destroy"


def test_one_by_one(library):
    g, lib = library
    things = objects(g)
    while things:
        del things[0]
    gc.collect()
    assert sorted(released(lib)) == FREED and released(lib)[-1] == "modp_ctx_destroy"
