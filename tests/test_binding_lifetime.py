"""Networks and batches are destroyed before the contexts they work on, in
whatever order the collector finalizes the Python objects (CPU: the library is
a stub that records its calls)."""
import ctypes as C
import gc

import pytest


class Stub:
    def __init__(self):
        self.calls, self.next = [], 1

    def __getattr__(self, name):
        if not name.startswith("iskra_"):
            raise AttributeError(name)

        def call(*a):
            if name.endswith("_create"):
                a[-1]._obj.value = self.next
                self.next += 1
            elif name.endswith("_destroy"):
                self.calls.append((name, a[0].value if isinstance(a[0], C.c_void_p) else a[0]))
            return 0
        return call


@pytest.mark.parametrize("how", ["collected", "context closed", "closed in order"])
@pytest.mark.parametrize("kind", ["network", "batch"])
def test_order(monkeypatch, how, kind):
    from iskra_amd import _lib as L
    stub = Stub()
    monkeypatch.setattr(L, "lib", lambda: stub)

    class Holder:
        pass
    h = Holder()
    h.me = h  # a cycle, as a traceback's frames make one
    h.ctx = L.Context(0)
    h.obj = L.WarmStart(h.ctx) if kind == "network" else L.Batch([h.ctx, L.Context(0)])
    if how == "context closed":
        h.ctx.close()
        assert not h.obj.h
    elif how == "closed in order":
        h.obj.close()
        h.ctx.close()
    del h
    gc.collect()
    names = [n for n, _ in stub.calls]
    own = "iskra_ws_destroy" if kind == "network" else "iskra_batch_destroy"
    assert names.count(own) == 1 and names[0] == own, names
    assert names.count("iskra_ctx_destroy") == (1 if kind == "network" else 2)
