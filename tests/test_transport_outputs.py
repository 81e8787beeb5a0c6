"""transport(check=False) of a call that fails before it writes: the arrays are zeros, not what the memory
held before."""
import numpy as np

from superlite_amd import slgpu


class Refusing:
    """a library whose transport returns an error and writes nothing"""
    def slgpu_transport(self, *args):
        return 5


def test_unchecked_failure_returns_zeros(monkeypatch):
    empty = np.empty

    def dirty(*args, **kw):
        a = empty(*args, **kw)
        a.fill(7)
        return a
    monkeypatch.setattr(slgpu.np, "empty", dirty)
    ctx = slgpu.Context.__new__(slgpu.Context)
    ctx.L, ctx.h, ctx.nx, ctx.ng = Refusing(), None, 3, 4
    r = ctx.transport(1, check=False)
    assert r["rc"] == 5
    for k, v in r.items():
        if k != "rc":
            assert np.all(np.asarray(v) == 0), k
