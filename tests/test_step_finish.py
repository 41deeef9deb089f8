"""The fill reports of a run of sweeps, read at its end by one kernel: directly
(up to 2048 tiles) or through a first reduction per sweep (more).  With u = 0
the sweeps leave f alone, except that cleanWisp! cuts an overfilled cell to 1
after the first of them, so exactly one sweep reports: the value and the flat
index of the cell (the first of two equal ones), at either extreme."""
import numpy as np
import pytest

from __graft_entry__ import load_package
from test_gpu_parity import say

pytestmark = pytest.mark.gpu

ia = load_package()


@pytest.mark.parametrize("T", [np.float32, np.float64])
@pytest.mark.parametrize("dims", [(64, 64), (500, 36), (1024, 640), (24, 20, 16), (128, 128, 136)])
def test_fill_report(dims, T):
    say("fill report", dims, T.__name__)
    s = ia.TwoPhaseSimulation(dims, (0.0,) * len(dims), float(dims[0]), T=T)
    f = np.asfortranarray(np.full(s.Ng, 0.25, dtype=T))
    s.intf.f = f
    st = ia.advect_(s, dt=0.25)
    assert st.status == 0 and st.fill_warnings == 0 and abs(st.vol - 0.25 * np.prod(dims)) <= 1e-9 * np.prod(dims)
    for val, name in ((1.5, "max"), (-0.5, "min")):
        g = f.copy(order="F")
        a, b = tuple(n - 3 for n in s.Ng), tuple(n - 2 for n in s.Ng)
        g[a] = g[b] = val
        s.intf.f = g
        st = ia.advect_(s, dt=0.25)
        msg = s._lib.ia_last_error(s._ctx).decode()
        idx = int(np.ravel_multi_index(a, s.Ng, order="F"))
        assert st.status == 3 and st.fill_warnings == 1
        assert f"{name} {val:.9g} @ {idx}" in msg, (msg, idx)
    g = f.copy(order="F")
    g[a] = np.nan
    s.intf.f = g
    with pytest.raises(ia.IAError) as e:
        ia.advect_(s, dt=0.25)
    assert e.value.code == 1
    s.close()
