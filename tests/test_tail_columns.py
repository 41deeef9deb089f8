"""The one-workgroup tail of the V-cycle with its cells in columns (FP32)
against the FP32 oracle, which runs the levels one by one: the default
solver's projections (6 pcg! iterations a level) on grids whose tail levels
are 512 threads of 4 or 8 cells, 1024 of 4, or do not fit columns at all, with
columns that the cells do not fill, sides that halve to odd ones and periodic
axes.  Both sides do the same operations per cell in FP32 and round FP64 sums
to FP32; the bars are those of the FP32 projection tests."""
import ctypes as C

import numpy as np
import pytest

from __graft_entry__ import load_package
from oracle import oracle as O
from test_gpu_parity import say

pytestmark = pytest.mark.gpu

ia = load_package()


@pytest.mark.parametrize("dims,perdir", [
    ((32, 32, 32), ()), ((32, 32, 32), (1, 2, 3)), ((64, 64), ()), ((128, 128), (1,)), ((60, 44), (2,)),
    ((44, 36, 20), (1,)), ((36, 20, 28), (3,)), ((40, 40, 20), ()), ((24, 24, 16), (2,)), ((96, 64), ()),
    ((40, 16, 48), (1, 3)), ((16, 8, 8), ()),
])
def test_projection_matches_oracle(dims, perdir):
    D = len(dims)
    say("tail in columns", dims, perdir)
    kw = dict(T=np.float32, perdir=perdir, λρ=1e-2)
    g = ia.TwoPhaseSimulation(dims, (0.0,) * D, float(dims[-1]), poisson_tol=1e-3, poisson_itmx=8, **kw)
    o = O.OracleSim(dims, (0.0,) * D, float(dims[-1]), mg_tol=1e-3, mg_itmx=8, **kw)
    x = np.meshgrid(*[(np.arange(n + 2) - 0.5) / n for n in dims], indexing="ij")
    f = (0.5 + 0.5 * np.tanh(8 * np.cos(2 * np.pi * x[0]) * np.cos(2 * np.pi * x[D - 1]))).astype(np.float32)
    rng = np.random.default_rng(5)
    u = (0.5 * rng.standard_normal(tuple(n + 2 for n in dims) + (D,))).astype(np.float32)
    for a in range(D):
        for i in range(D):
            v = u[..., i]
            ix = lambda s, a=a: tuple(s if b == a else slice(None) for b in range(D))  # noqa: E731
            if a + 1 in perdir:
                v[ix(0)], v[ix(-1)] = v[ix(-2)], v[ix(1)]
            elif a == i:
                for s in (0, 1, -1):
                    v[ix(s)] = 0
    for name, val in (("f", f), ("f0", f)):
        setattr(g.intf, name, val)
    g.flow.u = u
    o.set(O.F, np.asfortranarray(f))
    o.set(O.F0, np.asfortranarray(f))
    o.set(O.U, np.asfortranarray(u))
    g._call("ia_update_L", 0)
    g._call("ia_mg_update")
    o.lib.oc_update_L(o.ctx, 0)
    o.lib.oc_mg_update(o.ctx)
    st = ia.IASolveStats()
    g._call("ia_project", 0.5, C.byref(st))
    it, r2 = o.project(0.5)
    du = np.abs(g.flow.u.astype(np.float64) - o.u).max() / np.abs(o.u).max()
    pg, po = O.inside(g.flow.p).astype(np.float64), O.inside(o.p).astype(np.float64)
    dp = np.abs(pg - po).max() / np.abs(po).max()
    print(f"{dims} {perdir}: V-cycles {st.iters} / {it}, Δu {du:.2e}, Δp {dp:.2e}")
    assert abs(st.iters - it) <= 1
    assert du <= 2e-3 and dp <= 2e-3
    g.close()
