"""The transport against the oracle particle by particle where its per-cell records and its short
DDMC step change course: cell counts around a block of the records' kernel, expanding and
contracting meshes (Doppler shifts up and down in group, at the first and last group too), few
groups, with and without the amplification factor (a kernel of its own), walks cut off in the middle.

The walk is decided by comparisons of the same numbers, so the discrete outcome of every particle is
the oracle's; energies are products of at most 3000 factors and a few frame changes, each within
2^-52 or two of the oracle's: 1e-11."""
import numpy as np
import pytest

from oracle import pyoracle as po
from test_gpu_lines64 import GAS, IZ, II, problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ng,steps", [(2, 5, 3000), (3, 40, 3000), (64, 33, 1500), (255, 60, 700), (256, 61, 700),
                                         (257, 300, 700)])
@pytest.mark.parametrize("sign", [1.0, -1.0])
@pytest.mark.parametrize("ampfact", [False, True])
def test_transport_sizes(tables, nx, ng, steps, sign, ampfact):
    from superlite_amd import slgpu as S
    print("case: transport sizes", nx, ng, steps, sign, ampfact, flush=True)
    wl, lines, st = problem(nx, ng, 40 * ng, 6000.0, 7 * nx + ng)
    st["mass"][:] = 1.0
    nep = int(np.rint(np.sqrt(ng)))
    nepg = -(-ng // (nep + 1))
    n = 600
    ctx = S.Context(nx, ng, nep, nepg, npartmax=n, seed=9, max_steps=steps, errorfatal=False, ampfact=ampfact)
    ctx.set_groups(wl)
    ctx.set_ions(IZ, II)
    ctx.set_tables(*tables)
    ctx.set_lines(*lines)
    g = ctx.opacity_build(*[st[k] for k in GAS])
    # shells about as thick as the two optical-depth limits: IMC, unlumped and lumped groups in one cell
    x = np.cumsum(np.concatenate([[4.0], 7.0 / np.median(g["cap"], axis=1)]))
    vol = 4.0 / 3.0 * np.pi * np.diff(x ** 3)
    t = x[-1] / 1.5e9
    vx = x / t if sign > 0 else (x[-1] - x) / t
    divv = np.full(nx, sign * 3.0 / t)
    ctx.set_grid(x, vx, divv, vol, 0.5 * (x[1:] + x[:-1]))
    p = ctx.ddmc_prep(st["temp"], 1e43)
    nvol, nnew = ctx.sources(n, 3)
    tr = ctx.transport(3, check=False)
    q = ctx.particles(nnew)
    ctx.close()
    m = po.Model(x, vx, divv, vol, wl, nep, nepg, g["cap"], g["sig"], g["capgrey"], 1.0 / st["temp"], st["temp"],
                 tauddmc=5.0, taulump=10.0, max_steps=steps, ampfact=ampfact)
    m.set(opaclump=p["opaclump"], emitprob=p["emitprob"], emit=p["emit"], nvol=nvol)
    o = m.iteration(9, 3, per_particle=True)
    op = o["particles"]
    print("steps imc, ddmc, longest, errors", tr["nstepimc"], tr["nstepddmc"], tr["nstepmax"], tr["nerr"], flush=True)
    for k in ("stat", "ig", "nstep"):
        assert np.array_equal(q[k], op[k]), k
    for k in ("nstepimc", "nstepddmc", "nflux", "nerr"):
        assert tr[k] == o[k], k
    np.testing.assert_allclose(q["e"], op["e"], rtol=1e-11)
    np.testing.assert_allclose(tr["tally"], o["tally"], rtol=1e-11, atol=1e-11 * o["tally"].max())
