"""The DDMC preparation at the sizes where its kernels change course: rows shorter than, equal to
and just past a tile of the running sums, cell counts that do not fill a block of rows, rows
past the CU's LDS (the searches then run on global memory), a single lumped or unlumped group.

Against the oracle: leakage opacities and emission probabilities to 1e-12 (the sums' order
differs from the oracle's only inside the leakage sums), the sources' groups, and the bucket
maps against the plain searches for every draw."""
import numpy as np
import pytest

from oracle import pyoracle as po

from test_gpu_lines64 import GAS, IZ, II, problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ng,nline", [(3, 5, 60), (9, 255, 900), (8, 256, 900), (7, 257, 900),
                                         (17, 513, 2000), (16, 1025, 4000), (2, 20100, 9000)])
def test_prep_sizes(tables, nx, ng, nline):
    from superlite_amd import slgpu as S
    print("case: ddmc prep sizes", nx, ng, nline, flush=True)
    wl, lines, st = problem(nx, ng, nline, 6000.0, 5 * nx + ng)
    st["mass"][:] = 1.0
    nep = int(np.rint(np.sqrt(ng)))
    nepg = -(-ng // (nep + 1))
    ctx = S.Context(nx, ng, nep, nepg, npartmax=4096, seed=5)
    ctx.set_groups(wl)
    ctx.set_ions(IZ, II)
    ctx.set_tables(*tables)
    ctx.set_lines(*lines)
    g = ctx.opacity_build(*[st[k] for k in GAS])
    # shells about as thick as the lump threshold, so that cells hold lumped and unlumped groups
    x = np.cumsum(np.concatenate([[0.0], 12.0 / np.median(g["cap"], axis=1)]))
    vol = 4.0 / 3.0 * np.pi * np.diff(x ** 3)
    st.update(xarr=x, vxarr=x / 1.7e6, divv=np.full(nx, 3.0 / 1.7e6), rcell=0.5 * (x[1:] + x[:-1]))
    ctx.set_grid(x, st["vxarr"], st["divv"], vol, st["rcell"])
    p = ctx.ddmc_prep(st["temp"], 1e43)
    m = po.Model(x, st["vxarr"], st["divv"], vol, wl, nep, nepg, g["cap"], g["sig"], g["capgrey"],
                 1.0 / st["temp"], st["temp"], tauddmc=5.0, taulump=10.0)
    ol = m.leakage()
    for k in (0, 1, 6, 7, 9, 10):
        np.testing.assert_allclose(p["opaclump"][:, k], ol[:, k], rtol=1e-12, atol=0, err_msg=str(k))
    np.testing.assert_allclose(p["emitprob"], m.emission_probability(), rtol=1e-12)
    K = 1 << 14
    rng = np.random.default_rng(3)
    b = rng.integers(0, K, 700).astype(np.float64)
    r = np.concatenate([rng.random(3000), b / K, np.nextafter((b + 1) / K, 0.0), np.nextafter(b / K, 1.0), [1.0]])
    r = r[(r > 0.0) & (r <= 1.0)]
    rr, cc = np.tile(r, nx), np.repeat(np.arange(1, nx + 1), len(r)).astype(np.int32)
    for t in range(5):
        a, ref = ctx.sample_groups(t, rr, cc), ctx.sample_groups(t, rr, cc, direct=True)
        assert np.array_equal(a, ref), t
        assert (a <= ng).all() and (a[(a != 0) | (t == 4)] >= 1).all()
    m.set(opaclump=p["opaclump"], emitprob=p["emitprob"], emit=p["emit"])
    nvol, nnew = ctx.sources(4096, 3)
    m.set(nvol=nvol)
    o, q = m.sources(5, 3), ctx.particles(nnew)
    # a draw within rounding of an edge of the source spectrum may take the neighbouring group
    assert np.count_nonzero(~np.isclose(q["wl"], o["wl"], rtol=1e-13)) <= 1
    np.testing.assert_allclose(q["x"], o["x"], rtol=1e-13)
    ctx.close()
