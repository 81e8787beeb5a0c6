"""The FP64 opacity build's line sums (per-cell exponential tables and a short polynomial) at
the edges of their dispatch, against the CPU oracle and, for the backward, against the
unstaged kernels: polynomial degrees 6, 8 and 10 and the exp() form below them by temperature,
1, 4 and 16 waves per group by grid size, cells and groups that do not fill a block, line
counts that do not fill a trip, and a list with a negative level (no tables).

Tolerance 1e-12: the oracle's and the unstaged kernels' exponent product chi hc/kT <= 600 is rounded
to 2^-53, a relative error of its exponential of 7e-14; the sums and table entries add a few
units of 1e-16."""
import numpy as np
import pytest

from oracle import pyoracle as po
from superlite_amd import synth

pytestmark = pytest.mark.gpu

IZ = np.array([1, 2, 2, 8, 8, 8, 26, 26], np.int32)
II = np.array([1, 1, 2, 1, 2, 3, 1, 2], np.int32)


def problem(nx, ng, nline, temp, seed, negative=False):
    rng = np.random.default_rng(seed)
    wl = 1000e-8 * 32.0 ** (np.arange(ng + 1) / ng)
    k = rng.integers(0, len(IZ), nline)
    chi = rng.uniform(0.0, 80000.0, nline).astype(np.float32)
    if nline:
        chi[0] = 80655.0
        if negative:
            chi[-1] = -5.0
    lines = (np.sort(rng.uniform(990.0, 32100.0, nline)).astype(np.float32),
             (10.0 ** rng.normal(-4.0, 1.5, nline)).astype(np.float32), chi,
             IZ[k].astype(np.int16), II[k].astype(np.int16))
    oc = 10.0 ** rng.uniform(0.0, 8.0, (nx, len(IZ)))
    oc[rng.random(oc.shape) < 0.1] = 0.0
    fr = np.zeros((30, nx))
    for z, f in ((1, 0.4), (2, 0.2), (8, 0.3), (26, 0.1)):
        fr[z - 1] = f
    st = dict(temp=temp * rng.uniform(1.0, 1.2, nx), natom=1e53 * rng.uniform(0.5, 2.0, nx),
              vol=1e44 * rng.uniform(0.5, 2.0, nx), mass=np.ones(nx), nelec=rng.uniform(0.1, 1.5, nx),
              natomfr=fr, oc=oc, ginv=np.full(oc.shape, 0.5))
    st["mass"][nx // 2] = 0.0 if nx > 2 else 1.0
    return wl, lines, st


def context(S, nx, ng, wl, lines, tables):
    ctx = S.Context(nx, ng, 2, ng // 2 + 1, npartmax=16)
    x = 1e14 * np.arange(nx + 1)
    ctx.set_grid(x, x / 1.7e6, np.full(nx, 1.7e-6), 4.19 * np.diff(x ** 3), 0.5 * (x[1:] + x[:-1]))
    ctx.set_groups(wl)
    ctx.set_ions(IZ, II)
    ctx.set_tables(*tables)
    ctx.set_lines(*lines)
    return ctx


GAS = ("temp", "natom", "vol", "mass", "nelec", "natomfr", "oc", "ginv")


@pytest.mark.parametrize("nx,ng,nline,temp,negative", [
    (3, 5, 63, 6000.0, False), (64, 17, 400, 3300.0, False), (65, 1030, 5000, 5000.0, False),
    (130, 2800, 9001, 8000.0, False), (64, 16, 1, 9000.0, False), (65, 15, 0, 6000.0, False),
    (7, 20, 301, 2600.0, False), (66, 31, 500, 900.0, False), (5, 33, 777, 750.0, False),
    (65, 18, 402, 330.0, False), (4, 9, 200, 200.0, False), (6, 12, 150, 6000.0, True)])
def test_line_sums(tables, nx, ng, nline, temp, negative):
    from superlite_amd import slgpu as S
    print("case: fp64 line sums", nx, ng, nline, temp, negative, flush=True)
    wl, lines, st = problem(nx, ng, nline, temp, nx + ng, negative)
    ctx = context(S, nx, ng, wl, lines, tables)
    o = ctx.opacity_build(*[st[k] for k in GAS])
    ref = po.opacity(wl, st["temp"], st["natom"], st["vol"], st["mass"], st["nelec"], st["natomfr"],
                     IZ, II, st["oc"], st["ginv"], lines, tables)
    np.testing.assert_allclose(o["cap64"], ref["cap64"], rtol=1e-12, atol=0)
    rng = np.random.default_rng(1)
    g = [rng.standard_normal((nx, ng)) / max(np.abs(o["cap64"]).max(), 1e-300),
         rng.standard_normal(nx), rng.standard_normal(nx)]
    a = ctx.opacity_vjp(*g)
    ctx.set_unstaged(True)
    ctx.opacity_build(*[st[k] for k in GAS])
    b = ctx.opacity_vjp(*g)
    for k in a:
        scale = np.abs(b[k]).max()
        assert np.abs(a[k] - b[k]).max() <= 1e-12 * scale, k
    ctx.close()
