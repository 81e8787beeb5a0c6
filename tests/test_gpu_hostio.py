"""The outputs' way to the host (pinned chunks of 2 MiB, copying threads from 1 MiB on): sizes below,
at and across a chunk, more chunks than the ring has, arrays requested alone and together, into
ordinary and pinned memory, and two contexts in two threads.  Bytes are copied, so every
comparison is exact."""
import ctypes
import threading

import numpy as np
import pytest

from test_gpu_lines64 import GAS, context, problem

pytestmark = pytest.mark.gpu

WANT = ("cap64", "cap", "emiss", "sig", "capgrey", "capross")


def build(S, nx, ng, tables, seed=0):
    wl, lines, st = problem(nx, ng, 500, 6000.0, nx + seed)
    ctx = context(S, nx, ng, wl, lines, tables)
    return ctx, [st[k] for k in GAS]


# 1 MiB of doubles is 131072: one and two workers' shares, a full chunk (262144), one more, the ring's
# 12 MiB and beyond
@pytest.mark.parametrize("nx,ng", [(1, 5), (3, 777), (64, 2047), (64, 2048), (65, 2049), (64, 4096), (64, 4097),
                                   (127, 8190), (333, 9001)])
def test_outputs_alone_and_together(tables, nx, ng):
    import torch
    from superlite_amd import slgpu as S
    print("case: outputs", nx, ng, flush=True)
    ctx, gas = build(S, nx, ng, tables)
    full = ctx.opacity_build(*gas)
    for k in WANT:
        one = ctx.opacity_build(*gas, want=(k,))
        assert list(one) == [k] and np.array_equal(one[k], full[k])
    # pinned memory, which the GPU writes itself, and a misaligned place in ordinary memory
    keep = [np.ascontiguousarray(x if n != "natomfr" else np.asarray(x).T, np.float64) for n, x in zip(GAS, gas)]
    g = S.Gas(*[S._p(x) for x in keep])
    pinned = torch.full((nx, ng), -1.0, dtype=torch.float64, pin_memory=True)
    raw = np.full(4 * nx * ng + 9, 7, np.uint8)
    off = 8 - raw.ctypes.data % 8 + 4
    off = off if off + 4 * nx * ng < len(raw) else 4
    ctx._check(ctx.L.slgpu_opacity_build(ctx.h, ctypes.byref(g), 0, ctypes.c_void_p(pinned.data_ptr()),
                                         ctypes.c_void_p(raw.ctypes.data + off), None, None, None, None))
    assert np.array_equal(pinned.numpy(), full["cap64"])
    assert raw[off:off + 4 * nx * ng].tobytes() == full["cap"].tobytes()
    assert np.all(raw[:off] == 7) and np.all(raw[off + 4 * nx * ng:] == 7)
    ctx.close()


def test_two_contexts_in_two_threads(tables):
    from superlite_amd import slgpu as S
    print("case: two contexts", flush=True)
    made = [build(S, 80 + 10 * t, 6000, tables, t) for t in range(2)]
    first = [c.opacity_build(*gas) for c, gas in made]
    bad = []

    def work(t):
        for _ in range(3):
            r = made[t][0].opacity_build(*made[t][1])
            bad.extend(k for k in WANT if not np.array_equal(r[k], first[t][k]))
    ts = [threading.Thread(target=work, args=(t,)) for t in range(2)]
    for t in ts: t.start()
    for t in ts: t.join()
    for c, _ in made: c.close()
    assert not bad
