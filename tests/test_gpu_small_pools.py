"""Small particle pools: what a launch costs does not grow with the lanes it leaves empty, and lanes of
pure IMC are not spread over more waves than help them.  On an MI355X the transport kernel took 112 us
for 50 particles of one step each with 2048 blocks, 20 us with the blocks that take particles; 300
particles of 3000 pure IMC steps took 0.9 of the time of 10^5 spread over all waves, 0.55 by 32 a wave.
The limits lie midway."""
import dataclasses

import numpy as np
import pytest

from superlite_amd import synth

pytestmark = pytest.mark.gpu


def kernel_ms(S, tables, nx, ng, nline, npart, **kw):
    w = dataclasses.replace(synth.WORKLOADS["c1"], ng=ng, nline=nline)
    st = synth.load_state("c1")
    iz, ii = st["ion_iz"], st["ion_ii"]
    lines = synth.line_list(w, iz, ii)
    c = slice(0, nx)
    nep = max(1, int(np.rint(np.sqrt(ng))))
    ctx = S.Context(nx, ng, nep, -(-ng // nep), npartmax=npart, errorfatal=False, **kw)
    ctx.set_grid(st["xarr"][:nx + 1], st["vxarr"][:nx + 1], st["divv"][c], st["vol"][c], st["rcell"][c])
    ctx.set_groups(synth.group_grid(w))
    ctx.set_ions(iz, ii)
    ctx.set_tables(*tables)
    ctx.set_lines(*lines)
    per_cell = [np.asarray(st[k])[c] for k in ("temp", "natom", "vol", "mass", "nelec")]
    ctx.opacity_build(*per_cell, np.asarray(st["natomfr"])[:, c], st["oc"][c], st["ginv"][c], want=())
    ctx.ddmc_prep(per_cell[0], w.lbol, want=False)
    t = []
    for _ in range(7):
        ctx.sources(npart, 1)
        ctx.timers(reset=True)
        r = ctx.transport(1, want=False, check=False)
        t.append(ctx.timers()["transport_kernel"])
    ctx.close()
    return min(t), r


def test_blocks_that_take_particles(tables):
    from superlite_amd import slgpu as S
    print("case: 50 particles", flush=True)
    for precision in (S.SLGPU_FP64, S.SLGPU_MIXED):
        t, r = kernel_ms(S, tables, 1, 2, 100, 50, precision=precision, max_steps=1)
        assert r["nactive"] == 50 and t < 0.060, t


def test_pure_imc_fills_half_waves(tables):
    from superlite_amd import slgpu as S
    print("case: pure IMC, small pool", flush=True)
    few, _ = kernel_ms(S, tables, 20, 300, 10_000, 300, puretran=True, max_steps=3000)
    many, r = kernel_ms(S, tables, 20, 300, 10_000, 100_000, puretran=True, max_steps=3000)
    assert r["nstepddmc"] == 0 and few < 0.72 * many, (few, many)
