"""The particles' way to the host: many particles on a small grid take no longer than on a large one (the
bytes are the same; pinned chunks sized by the small grid took a hundred times as long), and every
array arrives whole at counts around the ring's chunks."""
import time

import numpy as np
import pytest

from test_gpu_lines64 import GAS, IZ, II, problem

pytestmark = pytest.mark.gpu

N = 1_000_000


def sourced(S, nx, ng, tables, n):
    wl, lines, st = problem(nx, ng, 200, 6000.0, 4)
    st["mass"][:] = 1.0
    ctx = S.Context(nx, ng, 2, ng // 2 + 1, npartmax=n)
    ctx.set_groups(wl)
    ctx.set_ions(IZ, II)
    ctx.set_tables(*tables)
    ctx.set_lines(*lines)
    g = ctx.opacity_build(*[st[k] for k in GAS])
    x = np.cumsum(np.concatenate([[0.0], 12.0 / np.median(g["cap"], axis=1)]))
    ctx.set_grid(x, x / 1.7e6, np.full(nx, 3.0 / 1.7e6), 4.0 / 3.0 * np.pi * np.diff(x ** 3), 0.5 * (x[1:] + x[:-1]))
    ctx.ddmc_prep(st["temp"], 1e43)
    ctx.sources(n, 1)
    return ctx


def test_small_grid_is_no_slower(tables):
    from superlite_amd import slgpu as S
    print("case: particles of a small and a large grid", flush=True)
    best = {}
    for nx, ng in ((4, 16), (400, 1000)):
        ctx = sourced(S, nx, ng, tables, N)
        t = []
        for _ in range(5):
            t0 = time.perf_counter()
            ctx.particles()
            t.append(time.perf_counter() - t0)
        best[nx] = min(t)
        ctx.close()
    assert best[4] < 2.0 * best[400], best


@pytest.mark.parametrize("n", [1, 100, 262_143, 262_145, N])
def test_particles_whole(tables, n):
    from superlite_amd import slgpu as S
    print("case: particles", n, flush=True)
    ctx = sourced(S, 4, 16, tables, n)
    p = ctx.particles()
    q = ctx.particles(n // 2)
    r = ctx.particles()
    ctx.close()
    for k in p:
        assert np.array_equal(p[k], r[k]) and np.array_equal(p[k][:n // 2], q[k]), k
    assert np.all(np.isfinite(p["x"]) & (p["x"] > 0.0) & (p["e"] > 0.0) & (p["wl"] > 0.0) & (np.abs(p["mu"]) <= 1.0))
