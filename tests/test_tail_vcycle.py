"""One V-cycle against the FP32 oracle, whose tail runs level by level: the
finer levels have no later V-cycle to damp an error of the tail's columns (one
column end, one periodic face, one partly filled column).  Per cell both sides
do the same FP32 operations; their dot products add in another order in FP64
before they are rounded to FP32, which changes a rounding about once in 2^29
sums, here some 10^3 sums a case.  So the pressures agree but for the last
operations on p (scaling by the time step, the periodic images): a few 2^-24 of
its largest value; the bar is 1e-5 of it.  The default solver takes 512 threads
of 4 cells or 1024 of 4 (6 iterations a level), the flexible CG 512 of 8 where
4 do not hold the level (64 iterations a level)."""
import ctypes as C

import numpy as np
import pytest

from __graft_entry__ import load_package
from oracle import oracle as O
from test_gpu_parity import say

pytestmark = pytest.mark.gpu

ia = load_package()


@pytest.mark.parametrize("poisson", ["reference", "refined"])
@pytest.mark.parametrize("dims,perdir", [
    ((32, 32, 32), ()), ((32, 32, 32), (1, 2, 3)), ((64, 64), ()), ((128, 128), (1,)), ((60, 44), (2,)),
    ((44, 36, 20), (1,)), ((36, 20, 28), (3,)), ((40, 40, 20), ()), ((24, 24, 16), (2,)), ((96, 64), ()),
    ((40, 16, 48), (1, 3)), ((16, 8, 8), ()),
])
def test_one_vcycle(dims, perdir, poisson):
    D = len(dims)
    say("one V-cycle", dims, perdir, poisson)
    kw = dict(T=np.float32, perdir=perdir, λρ=1e-2)
    g = ia.TwoPhaseSimulation(dims, (0.0,) * D, float(dims[-1]), poisson=poisson, poisson_tol=1e-30, poisson_itmx=1,
                              poisson_rtol=1e-30, poisson_max_outer=1, **kw)
    o = O.OracleSim(dims, (0.0,) * D, float(dims[-1]), mg_tol=1e-30, mg_itmx=1, **kw)
    x = np.meshgrid(*[(np.arange(n + 2) - 0.5) / n for n in dims], indexing="ij")
    f = (0.5 + 0.5 * np.tanh(8 * np.cos(2 * np.pi * x[0]) * np.cos(2 * np.pi * x[D - 1]))).astype(np.float32)
    u = (0.5 * np.random.default_rng(7).standard_normal(tuple(n + 2 for n in dims) + (D,))).astype(np.float32)
    for a in range(D):
        for i in range(D):
            v = u[..., i]
            ix = lambda s, a=a: tuple(s if b == a else slice(None) for b in range(D))  # noqa: E731
            if a + 1 in perdir:
                v[ix(0)], v[ix(-1)] = v[ix(-2)], v[ix(1)]
            elif a == i:
                for s in (0, 1, -1):
                    v[ix(s)] = 0
    for name in ("f", "f0"):
        setattr(g.intf, name, f)
    g.flow.u = u
    for fid, val in ((O.F, f), (O.F0, f), (O.U, u)):
        o.set(fid, np.asfortranarray(val))
    g._call("ia_update_L", 0)
    g._call("ia_mg_update")
    o.lib.oc_update_L(o.ctx, 0)
    o.lib.oc_mg_update(o.ctx)
    st = ia.IASolveStats()
    g._call("ia_project", 0.5, C.byref(st))
    it = o.project(0.5)[0] if poisson == "reference" else o.project_fcg(0.5, 1e-30, 1)[0]
    assert st.iters == it == 1
    pg, po = O.inside(g.flow.p).astype(np.float64), O.inside(o.p).astype(np.float64)
    dp, du = float(abs(pg - po).max() / abs(po).max()), float(abs(g.flow.u - o.u).max() / abs(o.u).max())
    print(f"Δp {dp:.2e}, Δu {du:.2e}")
    assert float(abs(po).max()) > 0 and dp <= 1e-5
    g.close()
