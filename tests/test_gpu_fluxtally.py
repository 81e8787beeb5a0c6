"""The flux tally against numpy's binning of the same particles, around the group count where the bins
no longer fit a block's LDS and at particle counts below, around and above a block's share.

Counts are equal; a bin's sum of at most 40000 positive numbers, added in any order, is within
40000 * 2^-53 < 1e-11 of the exact one."""
import numpy as np
import pytest

from test_gpu_lines64 import GAS, IZ, II, problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ng", [2, 250, 2299, 2300, 2301])
@pytest.mark.parametrize("n", [1, 1023, 1025, 40_000])
def test_fluxtally(tables, ng, n):
    from superlite_amd import slgpu as S
    print("case: flux tally", ng, n, flush=True)
    nx = 3
    wl, lines, st = problem(nx, ng, 4 * ng, 6000.0, ng)
    st["mass"][:] = 1.0
    nep = int(np.rint(np.sqrt(ng)))
    nepg = -(-ng // (nep + 1))
    ctx = S.Context(nx, ng, nep, nepg, npartmax=n, seed=9, max_steps=2000, errorfatal=False)
    ctx.set_groups(wl)
    ctx.set_ions(IZ, II)
    ctx.set_tables(*tables)
    ctx.set_lines(*lines)
    g = ctx.opacity_build(*[st[k] for k in GAS])
    x = np.cumsum(np.concatenate([[4.0], 1.0 / np.median(g["cap"], axis=1)]))
    t = x[-1] / 1.5e9
    ctx.set_grid(x, x / t, np.full(nx, 3.0 / t), 4.0 / 3.0 * np.pi * np.diff(x ** 3), 0.5 * (x[1:] + x[:-1]))
    ctx.ddmc_prep(st["temp"], 1e43, want=False)
    _, nnew = ctx.sources(n, 3)
    ctx.transport(3, check=False)
    q = ctx.particles(nnew)
    for _ in range(2):
        f = ctx.fluxtally()
        out = q["stat"] == 1
        b = np.clip(np.searchsorted(wl, q["wl"][out], side="right"), 1, ng) - 1
        assert np.array_equal(f["lumnum"], np.bincount(b, minlength=ng))
        for k, v in (("luminos", q["e"][out]), ("lumdev", q["e"][out] ** 2)):
            ref = np.zeros(ng, np.longdouble)
            np.add.at(ref, b, v.astype(np.longdouble))
            np.testing.assert_allclose(f[k], ref.astype(float), rtol=1e-11)
    ctx.close()
