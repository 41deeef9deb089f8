"""Ghost images written by kernels whose wavefronts are rows of cells: every
ghost entry holds what its boundary condition says, at row lengths around the
wavefront's and the tiles' edges, with the sides that are walls or periodic in
every mix.  Copies are exact, so the comparison is too."""
import itertools

import numpy as np
import pytest

from __graft_entry__ import load_package
from test_gpu_parity import say

pytestmark = pytest.mark.gpu

ia = load_package()

SHAPES = [(8, 8), (64, 12), (68, 8), (132, 64), (8, 8, 8), (64, 12, 8), (68, 8, 20), (128, 16, 72)]


def images(a, per):
    """The scalar with its ghosts rewritten, axis by axis, from its interior."""
    a = a.copy(order="F")
    for ax, p in enumerate(per):
        b = np.moveaxis(a, ax, 0)
        b[0], b[-1] = (b[-2], b[1]) if p else (b[1], b[-2])
    return a


def vec_images(u, per, ubc, exit_bc):
    u = u.copy(order="F")
    for i in range(len(per)):
        a, x1 = u[..., i], u[-1, ..., 0].copy(order="F")
        a = images(a, per)
        if not per[i]:
            b = np.moveaxis(a, i, 0)
            b[0] = b[1] = b[-1] = ubc[i]
        if exit_bc and i == 0:  # the exit face keeps its own value, its images copy that
            a[-1] = images(x1, per[1:])
        u[..., i] = a
    return u


@pytest.mark.parametrize("T", [np.float32, np.float64])
@pytest.mark.parametrize("dims", SHAPES)
def test_ghosts(dims, T):
    D = len(dims)
    rng = np.random.default_rng(sum(dims))
    for per in itertools.product((False, True), repeat=D):
        for exit_bc in (False,) if per[0] else (False, True):
            say("row images", dims, T.__name__, per, exit_bc)
            perdir = tuple(i + 1 for i in range(D) if per[i])
            ubc = tuple(0.0 if p else 0.125 * (i + 1) for i, p in enumerate(per))
            s = ia.TwoPhaseSimulation(dims, ubc, float(dims[0]), T=T, ν=0.01, λρ=0.1, perdir=perdir, exitBC=exit_bc)
            s.intf.f = images(np.asfortranarray(rng.uniform(0.05, 0.95, s.Ng).astype(T)), per)
            u = np.asfortranarray(rng.uniform(-0.1, 0.1, s.Ng + (D,)).astype(T))
            s.flow.u = vec_images(u, per, ubc, exit_bc)
            ia.MPFMomStep_(s, s, s)
            got = np.asarray(s.flow.u)
            assert np.isfinite(got).all()
            assert np.array_equal(got, vec_images(got, per, ubc, exit_bc))
            got = np.asarray(s.intf.f)
            assert np.array_equal(got, images(got, per))
            ls = ia.LevelSet(s)
            ia.redistaning_(ls, d=1, perdir=perdir)
            got = np.asarray(ls.ϕ)
            assert np.isfinite(got).all() and np.array_equal(got, images(got, per))
            s.close()
