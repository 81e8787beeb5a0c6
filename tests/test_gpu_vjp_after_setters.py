"""The FP64 backward after other lines or groups were set behind the build: it differentiates the
present line list at the built state, as the unstaged kernels do, which evaluate every line's
exponential from its record.  Lists with another top level (another step of the exponential tables),
the first of them without tables (a negative level) or the second, and the group setter, which sorts
the lines anew.

Tolerance 1e-12, as in test_gpu_lines64: exponent products up to 600 rounded to 2^-53, 7e-14, and a
few units of 1e-16 from sums and table entries."""
import numpy as np
import pytest

from test_gpu_lines64 import GAS, context, problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("change", ["lower top", "higher top", "tables after none", "none after tables", "groups"])
def test_backward_of_the_present_lines(tables, change):
    from superlite_amd import slgpu as S
    print("case: vjp after", change, flush=True)
    nx, ng = 65, 40
    wl, lines, st = problem(nx, ng, 900, 6000.0, 11)
    chi = lines[2]
    with_neg = chi.copy()
    with_neg[-1] = -5.0
    first, then = {"lower top": (chi, 0.4 * chi), "higher top": (chi, 2.0 * chi), "tables after none": (with_neg, chi),
                   "none after tables": (chi, with_neg), "groups": (chi, chi)}[change]
    ctx = context(S, nx, ng, wl, (*lines[:2], first.astype(np.float32), *lines[3:]), tables)
    o = ctx.opacity_build(*[st[k] for k in GAS])
    if change == "groups":
        # the line of the highest level falls off the grid: the tables' step is another one
        k = int(np.argmax(chi))
        assert wl[0] < lines[0][k] * 1e-8 < wl[-1]
        edge = np.linspace(lines[0][k] * 1e-8 * 1.001, wl[-1], ng + 1)
        assert chi[lines[0] * 1e-8 >= edge[0]].max() < 0.9999 * chi[k]
        ctx.set_groups(edge)
    else:
        ctx.set_lines(*lines[:2], then.astype(np.float32), *lines[3:])
    rng = np.random.default_rng(2)
    g = [rng.standard_normal((nx, ng)) / np.abs(o["cap64"]).max(), rng.standard_normal(nx), rng.standard_normal(nx)]
    a = ctx.opacity_vjp(*g)
    ctx.set_unstaged(True)
    b = ctx.opacity_vjp(*g)
    ctx.close()
    for k in a:
        assert np.abs(a[k] - b[k]).max() <= 1e-12 * np.abs(b[k]).max(), k
