"""NLTE populations and opacities at the edges of their dispatch: level counts around a wave's 64
rows, the largest whose matrix fits LDS (142) and the first that does not, and 1, 4 and 16 waves per
group of the line sums; a massless cell in each.

The populations are checked by their residual in the oracle's rate matrix, whose size does not
depend on the matrix's conditioning: |A x - b| <= 3 n 2^-53 |L| |U| |x| for the computed factors
(Higham, Accuracy and Stability of Numerical Algorithms, theorem 9.4), 5e-14 at n = 143, and the
exponents of the rates (up to 40 times 2^-53, a few operations) move A by some 1e-14: 1e-12.  The
row of ones is the last pivot of a matrix of up to 1e9, so its |L| |U| is larger than its |A|.  The opacities are compared with the per-line form on
the same populations: exponent products up to 600 rounded to 2^-53, 7e-14, and units of 1e-16 from
the sums: 1e-12."""
from functools import partial
from types import SimpleNamespace

import numpy as np
import pytest
import scipy.linalg

from oracle import pyoracle as po
from test_gpu_lines64 import GAS, IZ, II, context, problem

pytestmark = pytest.mark.gpu


def atom(n, rng):
    lev = np.arange(1, n + 1)
    chi, g = 109677.0 * (1.0 - 1.0 / lev ** 2), 2.0 * lev ** 2
    lo, hi = (x + 1 for x in np.triu_indices(n, 1))
    wl0 = 1e8 / (chi[hi - 1] - chi[lo - 1])
    f = 10.0 ** rng.uniform(-4.0, 0.0, len(lo))
    gl, gu = g[lo - 1], g[hi - 1]
    wf = wl0 * 1e-8
    fc = 0.02654
    aul = 8.0 * np.pi * fc * gl * f / (gu * wf ** 2)
    bul = 4.0 * np.pi * fc * wf * gl * f / (1.986e-16 * gu)
    blu = bul * gu / gl
    k = rng.permutation(len(lo))[:max(1, len(lo) // 2)]
    de = (chi[hi[k] - 1] - chi[lo[k] - 1]) / 8065.5
    c = np.stack([rng.normal(-1.0, 0.5, len(k)), rng.normal(0.0, 0.1, len(k)),
                  rng.normal(0.0, 0.02, len(k)), np.zeros(len(k))], 1)
    cl = lambda m: np.stack([rng.normal(m, 0.5, n), rng.normal(-0.5, 0.1, n), np.zeros(n), np.zeros(n)], 1)
    perm = rng.permutation(n)
    return dict(nlev=n, glev=g, llw=lo, lup=hi, wl0=wl0, f=f, gl=gl, gu=gu, aul=aul, bul=bul, blu=blu,
                llw_coll=lo[k], lup_coll=hi[k], coll_c=c, dele=de, lev_pi=lev[perm], pi_c=cl(1.0),
                rr_c=cl(-2.0), dele_pi=13.6 / lev[perm] ** 2)


@pytest.mark.parametrize("n,nx,ng,nline", [
    (2, 3, 5, 63), (3, 65, 40, 900), (37, 9, 33, 700), (63, 5, 20, 300), (64, 66, 1030, 5000), (65, 4, 50, 500),
    (100, 130, 2800, 9001), (128, 6, 64, 900), (129, 3, 30, 100), (142, 7, 25, 400), (143, 5, 31, 300)])
@pytest.mark.parametrize("mixed", [False, True])
def test_nlte_sizes(tables, n, nx, ng, nline, mixed):
    from superlite_amd import slgpu as S
    print("case: nlte sizes", n, nx, ng, nline, mixed, flush=True)
    rng = np.random.default_rng(n)
    wl, lines, st = problem(nx, ng, nline, 6000.0, n)
    sp = atom(n, rng)
    ndens = 10.0 ** rng.uniform(6.0, 10.0, (nx, 2))
    radtemp = 0.9 * st["temp"]
    args = [st[k] for k in GAS] + [radtemp, ndens]
    prec = S.SLGPU_MIXED if mixed else S.SLGPU_FP64
    ctx = context(SimpleNamespace(Context=partial(S.Context, precision=prec)), nx, ng, wl, lines, tables)
    ctx.set_nlte_data(sp)
    r = ctx.opacity_build_nlte(*args)
    ctx.set_unstaged(True)
    u = ctx.opacity_build_nlte(*args)
    ctx.close()
    assert np.array_equal(r["npop"], u["npop"])
    assert np.all(r["npop"][st["mass"] <= 0.0] == 0.0)
    gas = [wl] + [st[k] for k in GAS[:6]] + [IZ, II, st["oc"], st["ginv"], lines, tables]
    for i in {0, nx - 1}:
        a, b = po.nlte_rate_matrix(sp, radtemp, ndens, i, *gas)
        x = r["npop"][i]
        p, lo, up = scipy.linalg.lu(a)
        size = p @ (np.abs(lo) @ (np.abs(up) @ np.abs(x))) + np.abs(b)
        assert np.max(np.abs(a @ x - b) / size) < 1e-12
    # random populations can change sign: the terms' size is that of the largest
    for k, tol in (("cap64", 1e-12), ("emiss", 1.3e-7), ("capemit", 1.3e-7)):
        np.testing.assert_allclose(r[k], u[k], rtol=tol, atol=tol * np.abs(u[k]).max())
