"""The coarse CG and pcg! in one launch (ia_cgp.h) against one launch per iteration
(IA_CG1_NB set), which evaluates the same recurrence: whole projections to
1e-6 from the same inputs, on grids whose coarse levels meet every edge of
the boxes: levels that the boxes do not divide, sides of 2 cells, sides that
halve to odd ones, walls and periodic axes (a box that is its own neighbour
among them), and a level of so many workgroups that their sums are formed in
groups.  Per cell both do the same operations in the same order; their dot
products add in another order in FP64 before they are rounded to FP32, which
changes a rounding of 2^-24 about once in 2^29 sums.  The bar allows such
changes to reach the result at the size of the solve's tolerance."""
import ctypes as C
import os

import numpy as np
import pytest

from __graft_entry__ import load_package
from test_gpu_parity import say

pytestmark = pytest.mark.gpu

ia = load_package()


def projected(dims, perdir, launched, **kw):
    old = os.environ.get("IA_CG1_NB")
    if launched:
        os.environ["IA_CG1_NB"] = "256"
    try:
        s = ia.TwoPhaseSimulation(dims, (0.0,) * len(dims), float(dims[-1]), T=np.float32, perdir=perdir, **kw)
    finally:
        if launched:
            del os.environ["IA_CG1_NB"]
            if old is not None:
                os.environ["IA_CG1_NB"] = old
    rng = np.random.default_rng(11)
    D = len(dims)
    x = np.meshgrid(*[np.arange(n + 2) / n for n in dims], indexing="ij")
    f = 0.5 + 0.5 * np.tanh(20 * np.sin(2 * np.pi * x[0]) * np.cos(2 * np.pi * x[D - 1]))
    s.intf.f = f
    u = 0.1 * rng.standard_normal(tuple(n + 2 for n in dims) + (D,))
    for a in range(D):  # no flow through walls
        if a + 1 not in perdir:
            for q in (0, 1, -1):
                u[tuple(q if b == a else slice(None) for b in range(D)) + (a,)] = 0
        else:
            ix = [slice(None)] * D
            ix[a] = -1
            lo = [slice(None)] * D
            lo[a] = 1
            u[tuple(ix)] = u[tuple(lo)]
    s.flow.u = u
    s._call("ia_update_L", 0)
    s._call("ia_mg_update")
    st = ia.IASolveStats()
    s._call("ia_project", 1.0, C.byref(st))
    out = s.flow.u.astype(np.float64), s.flow.p.astype(np.float64), st.iters, st.rel, s.flow.σ.astype(np.float64), st.r2
    s.close()
    return out


@pytest.mark.parametrize("dims,perdir", [
    ((256, 200), ()), ((200, 136), (1, 2)), ((2048, 16), (2,)), ((16, 2048), (1,)),
    ((64, 64, 64), ()), ((120, 88, 72), (1, 2)), ((100, 60, 84), (3,)), ((512, 16, 16), (1, 2, 3)),
    ((16, 256, 32), ()), ((160, 160, 96), (2,)), ((240, 208, 200), (1,)), ((256, 256, 248), (3,)),
])
def test_one_launch_equals_one_launch_per_iteration(dims, perdir):
    say("coarse CG in one launch", dims, perdir)
    u, p, it, rel, _, _ = projected(dims, perdir, False, poisson="refined")
    ul, pl, itl, rell, _, _ = projected(dims, perdir, True, poisson="refined")
    print(f"iterations {it} / {itl}, rel {rel:.3e} / {rell:.3e}, max|Δu| {np.abs(u - ul).max():.2e}, "
          f"max|Δp| {np.abs(p - pl).max():.2e} of {np.abs(pl).max():.2e}")
    assert 0 < rel <= 1e-6 and abs(it - itl) <= 1
    assert np.abs(u - ul).max() <= 1e-5 * np.abs(ul).max()
    assert np.abs(p - pl).max() <= 1e-4 * np.abs(pl).max()


@pytest.mark.parametrize("dims,perdir", [
    ((64, 64), (1, 2)), ((256, 200), ()), ((1000, 24), (2,)), ((512, 512), ()), ((1024, 640), (1,)),
    ((48, 32, 40), ()), ((100, 60, 84), (1, 3)), ((64, 64, 64), ()), ((96, 96, 96), (2,)),
])
def test_default_solver_in_one_launch(dims, perdir):
    """pcg! on the finest and the coarse levels in one launch each against its
    launches, over three V-cycles of the default solver that it does not end
    earlier: u, p, the scratch that Flow.σ holds afterwards, and Σr² (FP64
    parts of FP32 values) to the bars above."""
    say("pcg! in one launch", dims, perdir)
    kw = dict(poisson="reference", poisson_tol=1e-12, poisson_itmx=3)
    u, p, it, _, z, r2 = projected(dims, perdir, False, **kw)
    ul, pl, itl, _, zl, r2l = projected(dims, perdir, True, **kw)
    print(f"Σr² {r2:.6e} / {r2l:.6e}, max|Δu| {np.abs(u - ul).max():.2e}, max|Δp| {np.abs(p - pl).max():.2e}")
    assert it == itl == 3
    assert abs(r2 - r2l) <= 1e-4 * r2l
    assert np.abs(u - ul).max() <= 1e-5 * np.abs(ul).max()
    assert np.abs(p - pl).max() <= 1e-4 * np.abs(pl).max()
    assert np.abs(z - zl).max() <= 1e-4 * np.abs(zl).max()


@pytest.mark.parametrize("poisson", ["refined", "reference"])
def test_contexts_take_the_xcds_in_turn(poisson):
    """Nine contexts, one after the other: wherever a launch runs, the same bits."""
    dims = (192, 136)
    say("one launch on each XCD", dims, poisson)
    ref = projected(dims, (), False, poisson=poisson)
    for _ in range(8):
        got = projected(dims, (), False, poisson=poisson)
        assert got[2] == ref[2] and all(np.array_equal(a, b) for a, b in zip((got[0], got[1]), (ref[0], ref[1])))
