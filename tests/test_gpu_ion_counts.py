"""The opacity build and its backward in FP64 at the ion counts where their kernels change, with cells the
exponential tables suit (6000 K) and cells too cold for them (250 K): populations staged in LDS beside
the tables (up to 240 ions in the build, any number the backward takes) or without them (up to 128 and
56), and unstaged beyond.  Against the CPU oracle and, for the backward, the unstaged kernels.

Tolerance 1e-12: at 80655 cm^-1 and 250 K the exponent product chi hc/kT is 464, rounded to 2^-53 in the
oracle, a relative error of its exponential of 5e-14; sums and table entries add a few units of 1e-16.

Cells without tables must not fall back to the unstaged kernels, which gather a population per line
(64 x 1000 groups x 1e5 lines: 45 us staged and 68 us unstaged, the backward 0.18 and 0.43 ms)."""
import numpy as np
import pytest

from oracle import pyoracle as po
from test_gpu_lines64 import GAS, problem

pytestmark = pytest.mark.gpu

ALL = np.array([(z, i) for z in range(1, 31) for i in range(1, z + 1)], np.int32)


def many_ions(nion, nx, ng, nline, temp):
    """problem()'s inputs with the first nion ions of the elements in order"""
    wl, lines, st = problem(nx, ng, nline, temp, nion)
    rng = np.random.default_rng(nion)
    iz, ii = ALL[:nion].T.copy()
    k = rng.integers(0, nion, nline)
    lines = (*lines[:3], iz[k].astype(np.int16), ii[k].astype(np.int16))
    st["oc"] = 10.0 ** rng.uniform(0.0, 8.0, (nx, nion))
    st["oc"][rng.random(st["oc"].shape) < 0.1] = 0.0
    st["ginv"] = np.full(st["oc"].shape, 0.5)
    return wl, lines, st, iz, ii


def context(S, nx, ng, wl, lines, tables, iz, ii):
    ctx = S.Context(nx, ng, 2, ng // 2 + 1, npartmax=16)
    x = 1e14 * np.arange(nx + 1)
    ctx.set_grid(x, x / 1.7e6, np.full(nx, 1.7e-6), 4.19 * np.diff(x ** 3), 0.5 * (x[1:] + x[:-1]))
    ctx.set_groups(wl)
    ctx.set_ions(iz, ii)
    ctx.set_tables(*tables)
    ctx.set_lines(*lines)
    return ctx


@pytest.mark.parametrize("nion", [56, 57, 124, 128, 129, 240, 241])
@pytest.mark.parametrize("nx,ng,nline,temp", [(66, 20, 2000, 6000.0), (3, 33, 1500, 250.0)])
def test_ion_counts(tables, nion, nx, ng, nline, temp):
    from superlite_amd import slgpu as S
    print("case: ion counts", nion, nx, ng, temp, flush=True)
    wl, lines, st, iz, ii = many_ions(nion, nx, ng, nline, temp)
    ctx = context(S, nx, ng, wl, lines, tables, iz, ii)
    o = ctx.opacity_build(*[st[k] for k in GAS])
    ref = po.opacity(wl, st["temp"], st["natom"], st["vol"], st["mass"], st["nelec"], st["natomfr"], iz, ii,
                     st["oc"], st["ginv"], lines, tables)
    np.testing.assert_allclose(o["cap64"], ref["cap64"], rtol=1e-12, atol=0)
    if nion + 4 <= 128:                                    # four elements; the backward's limit
        rng = np.random.default_rng(1)
        g = [rng.standard_normal((nx, ng)) / np.abs(o["cap64"]).max(), rng.standard_normal(nx), rng.standard_normal(nx)]
        a = ctx.opacity_vjp(*g)
        ctx.set_unstaged(True)
        b = ctx.opacity_vjp(*g)
        for k in a:
            assert np.abs(a[k] - b[k]).max() <= 1e-12 * np.abs(b[k]).max(), k
    ctx.close()


def test_cold_cells_stay_staged(tables):
    from superlite_amd import slgpu as S
    print("case: cold cells' kernels", flush=True)
    nx, ng = 64, 1000
    wl, lines, st, iz, ii = many_ions(8, nx, ng, 100_000, 250.0)
    ctx = context(S, nx, ng, wl, lines, tables, iz, ii)
    g = np.random.default_rng(2).standard_normal((nx, ng))
    ms = {}
    for unstaged in (False, True):
        ctx.set_unstaged(unstaged)
        t = []
        for _ in range(9):
            ctx.timers(reset=True)
            ctx.opacity_build(*[st[k] for k in GAS], want=("sig",))
            ctx.opacity_vjp(g)
            tm = ctx.timers()
            t.append((tm["opacity_kernel"], tm["opacity_vjp_kernels"]))
        ms[unstaged] = np.min(t, axis=0)
    ctx.close()
    assert np.all(ms[False] < [0.85, 0.7] * ms[True]), ms
