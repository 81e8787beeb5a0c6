"""The lumped rows' bucket maps against the plain searches at both ends of every one of the 2^14
buckets: the two agree on every draw between when they agree there, since both are steps that rise
with the draw.  Rows of a few groups up to several per bucket, in expanding and contracting meshes
(whose Doppler rows run the other way)."""
import numpy as np
import pytest

from test_gpu_lines64 import GAS, IZ, II, problem

pytestmark = pytest.mark.gpu

K = 1 << 14


@pytest.mark.parametrize("nx,ng", [(2, 2), (3, 5), (2, 1023), (2, 1024), (2, 1025), (2, 30_000)])
@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_bucket_ends(tables, nx, ng, sign):
    from superlite_amd import slgpu as S
    print("case: bucket ends", nx, ng, sign, flush=True)
    wl, lines, st = problem(nx, ng, 2 * ng, 6000.0, 5 * nx + ng)
    st["mass"][:] = 1.0
    nep = int(np.rint(np.sqrt(ng)))
    ctx = S.Context(nx, ng, nep, -(-ng // (nep + 1)), npartmax=64, seed=5)
    ctx.set_groups(wl)
    ctx.set_ions(IZ, II)
    ctx.set_tables(*tables)
    ctx.set_lines(*lines)
    g = ctx.opacity_build(*[st[k] for k in GAS])
    x = np.cumsum(np.concatenate([[0.0], 12.0 / np.median(g["cap"], axis=1)]))
    vx = x / 1.7e6 if sign > 0 else (x[-1] - x) / 1.7e6
    ctx.set_grid(x, vx, np.full(nx, sign * 3.0 / 1.7e6), 4.0 / 3.0 * np.pi * np.diff(x ** 3), 0.5 * (x[1:] + x[:-1]))
    ctx.ddmc_prep(st["temp"], 1e43)
    b = np.arange(K, dtype=np.float64)
    r = np.concatenate([b[1:] / K, np.nextafter((b + 1) / K, 0.0), [1.0]])
    rr, cc = np.tile(r, nx), np.repeat(np.arange(1, nx + 1), len(r)).astype(np.int32)
    for t in range(5):
        a, ref = ctx.sample_groups(t, rr, cc), ctx.sample_groups(t, rr, cc, direct=True)
        assert np.array_equal(a, ref), t
    ctx.close()
