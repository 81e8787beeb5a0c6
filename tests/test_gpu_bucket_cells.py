"""The bucket maps on both sides of the mesh size at which their kernel changes (24 cells by plain
searches, 25 by a block per map), against the plain searches at both ends of every bucket, as
test_gpu_bucket_maps does on small meshes: a map is exact when it agrees there.  The destinations'
flags in the entries are covered on both sides by test_gpu_transport_sizes, walk by walk."""
import numpy as np
import pytest

from test_gpu_lines64 import GAS, IZ, II, problem

pytestmark = pytest.mark.gpu

K = 1 << 14


@pytest.mark.parametrize("nx,ng", [(24, 50), (25, 2), (25, 5), (25, 1023), (26, 1024), (25, 1025), (25, 30_000)])
@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_bucket_ends(tables, nx, ng, sign):
    from superlite_amd import slgpu as S
    print("case: bucket ends by cells", nx, ng, sign, flush=True)
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
    for i in {1, 2, nx // 2, nx - 1, nx}:
        cell = np.full(len(r), i, np.int32)
        for t in range(5):
            assert np.array_equal(ctx.sample_groups(t, r, cell), ctx.sample_groups(t, r, cell, direct=True)), (t, i)
    ctx.close()
