"""Surface tension where a wavefront's interface cells are none, few, just as
many as share out its lanes, or all: planes of several tilts across rows of 64
and more cells, against the oracle at test_surface_tension_force's tolerance."""
import numpy as np
import pytest

from oracle import oracle as O
from test_gpu_parity import maxdiff, pair, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [np.float64, np.float32])
@pytest.mark.parametrize("dims,n", [
    ((72, 16), (0.03, 1.0)), ((72, 16), (0.11, 1.0)), ((72, 16), (0.4, 1.0)), ((72, 16), (1.0, 0.05)),
    ((72, 16, 8), (0.03, 1.0, 0.02)), ((72, 16, 16), (0.3, 1.0, 0.2)), ((8, 16, 24), (1.0, 0.07, 0.3)),
    ((72, 8, 16), (0.02, 0.05, 1.0)),
])
def test_planes(dims, n, T):
    D = len(dims)
    say("surface tension of a plane", dims, n, T.__name__)
    c = [0.5 * dims[a] + 0.17 * (a + 1) for a in range(D)]
    l = np.sqrt(sum(v * v for v in n))
    sdf = lambda x: sum(n[a] * (x[a] - c[a]) for a in range(D)) / l + 0.6 * np.sin(0.2 * x[0])
    g, o = pair(dict(dims=dims, u_BC=(0.0,) * D, L=float(dims[0]),
                     kw=dict(T=T, λρ=0.1, λμ=0.1, ν=0.01, η=0.05, InterfaceSDF=sdf)))
    g._call("ia_visc", 0)
    o.lib.oc_visc(o.ctx, 0)
    Fg, Fo = O.inside(g.flow.force, D), O.inside(o.get(O.FORCE), D)
    assert np.abs(Fo).max() > 0
    assert maxdiff(Fg, Fo) <= (1e-12 if T == np.float64 else 1e-5) * np.abs(Fo).max()
    g.close()
