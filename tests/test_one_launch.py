"""Coarse solves in one launch: which levels take that path, that it is the one
that runs, and what happens when a launch's workgroups do not run together.  A
lost workgroup is one that was not launched: the others wait out their bounded
wait (20 ms) and every kernel ends by itself."""
import ctypes as C
import threading

import numpy as np
import pytest

from __graft_entry__ import load_package
from test_abi import _c_layout
from test_gpu_parity import say

ia = load_package()

REST = 16  # ia_cgp.h CGP_REST


def box(dims, perdir=(), seed=11, **kw):
    """A simulation with a mixed density field and its multigrid coefficients, and a velocity to project."""
    s = ia.TwoPhaseSimulation(dims, (0.0,) * len(dims), float(dims[-1]), T=np.float32, perdir=perdir, **kw)
    D = len(dims)
    x = np.meshgrid(*[np.arange(n + 2) / n for n in dims], indexing="ij")
    s.intf.f = 0.5 + 0.5 * np.tanh(20 * np.sin(2 * np.pi * x[0]) * np.cos(2 * np.pi * x[D - 1]))
    u = 0.1 * np.random.default_rng(seed).standard_normal(tuple(n + 2 for n in dims) + (D,))
    for a in range(D):
        ix = lambda q, a=a: tuple(q if b == a else slice(None) for b in range(D)) + (a,)  # noqa: E731
        if a + 1 in perdir:
            u[ix(-1)] = u[ix(1)]
        else:
            for q in (0, 1, -1):
                u[ix(q)] = 0
    s._call("ia_update_L", 0)
    s._call("ia_mg_update")
    return s, np.asfortranarray(u.astype(np.float32))


def project(s, u):
    s.flow.u = u
    s.flow.p = np.zeros(u.shape[:-1], np.float32)
    st = ia.IASolveStats()
    s._call("ia_project", 1.0, C.byref(st))
    return s.flow.u.copy(), s.flow.p.copy(), st


def info(s, lose=0):
    o = ia.IAOneLaunchInfo()
    s._call("ia_one_launch", lose, C.byref(o))
    return o


def test_info_layout_matches_header(tmp_path):
    f = [n for n, *_ in ia.IAOneLaunchInfo._fields_]
    lay = _c_layout(tmp_path, {"ia_one_launch_info": f})
    assert lay[("ia_one_launch_info", "sizeof")] == C.sizeof(ia.IAOneLaunchInfo)
    for n in f:
        assert lay[("ia_one_launch_info", n)] == getattr(ia.IAOneLaunchInfo, n).offset


def test_bench_counts_the_path_that_ran():
    """A coarse level's bytes: of a whole solve where it is one launch, of a step
    where it is not (whatever its size), of neither where the record mixes both."""
    import bench

    o = ia.IAOneLaunchInfo()
    o.levels = 0b1010
    assert bench.bytes_per_cell("cg1_l1", o) == bench.BYTES_PER_CELL["cg1_l1"] == 28
    assert bench.bytes_per_cell("cg1_l2", o) == 56 and bench.bytes_per_cell("vof", o) == 21
    o.given_up = 1
    assert bench.bytes_per_cell("cg1_l3", o) is None and bench.bytes_per_cell("cg1_l2", o) == 56


def div2(u):
    """Σ(div u)² over the interior: what a projection left of the residual."""
    D = u.ndim - 1
    u = u.astype(np.float64)
    at = lambda a, lo, hi: tuple(slice(lo, hi) if b == a else slice(1, -1) for b in range(D)) + (a,)  # noqa: E731
    s = sum(u[at(a, 2, None)] - u[at(a, 1, -1)] for a in range(D))
    return float((s * s).sum())


@pytest.mark.gpu
@pytest.mark.parametrize("poisson", ["refined", "reference"])
@pytest.mark.parametrize("dims", [(192, 136), (64, 64, 48)])
def test_give_up_is_reported_and_tried_again(dims, poisson):
    """The projection in which a solve gives up reaches what it reaches otherwise,
    says what happened, the next ones go by one launch per iteration, and after
    them the one-launch solves are back with the bits they had before.  Two
    solutions to the relative tolerance differ by that size (the bar of
    test_coarse_cg.py); the default solver's Σr² must be that of the projected
    velocity, FP32's rounding of the residual (a few per cent of it at these
    tolerances) aside."""
    say("one-launch solve gives up", dims, poisson)
    s, u = box(dims, poisson=poisson, poisson_tol=1e-4)

    def check(uk, st):
        if poisson == "refined":
            assert 0 < st.rel <= 1e-6
            assert float(abs(uk - u0).max()) <= 1e-5 * float(abs(u0).max())
        else:
            assert st.r2 <= 1e-4 or st0.iters == st.iters == 200  # FP32 may hold Σr² above the tolerance
            assert abs(div2(uk) - st.r2) <= 0.25 * st.r2

    u0, p0, st0 = project(s, u)
    check(u0, st0)
    o = info(s)
    assert o.levels and o.solves > 0 and o.given_up == 0 and o.rest == 0
    n = o.solves
    info(s, lose=1)
    u1, _, st1 = project(s, u)
    o = info(s)
    assert o.given_up == 1 and o.rest == REST and o.solves > n
    assert b"did not run together" in s._lib.ia_last_error(s._ctx)
    check(u1, st1)
    n = o.solves
    for k in range(1, REST):
        uk, _, st = project(s, u)
        o = info(s)
        assert o.rest == REST - k and o.solves == n and o.given_up == 1
        check(uk, st)
    u2, p2, st2 = project(s, u)
    o = info(s)
    assert o.rest == 0 and o.solves > n and o.given_up == 1
    assert st2.iters == st0.iters and (u2 == u0).all() and (p2 == p0).all()
    info(s, lose=1)  # the second time costs twice the rest
    project(s, u)
    o = info(s)
    assert o.given_up == 2 and o.rest == 2 * REST
    s.close()


@pytest.mark.gpu
@pytest.mark.parametrize("dims,perdir", [((192, 136), ()), ((64, 64, 48), (2,)), ((96, 96, 96), ())])
def test_plain_multigrid_throws_a_cut_short_correction_away(dims, perdir):
    """Plain multigrid adds each V-cycle's correction as it is: the one whose
    solve gave up is left out, so one more V-cycle does (one of slack)."""
    say("plain multigrid, one-launch solve gives up", dims, perdir)
    s, u = box(dims, perdir, poisson="plain", λρ=0.1)
    u0, _, st0 = project(s, u)
    assert info(s).solves > 0 and 0 < st0.rel <= 1e-6
    info(s, lose=1)
    u1, _, st1 = project(s, u)
    o = info(s)
    print(f"V-cycles {st0.iters} / {st1.iters}, rel {st1.rel:.2e}, {st0.ms:.1f} / {st1.ms:.1f} ms")
    assert o.given_up == 1 and o.rest == REST
    assert 0 < st1.rel <= 1e-6 and st0.iters < st1.iters <= st0.iters + 2
    assert float(abs(u1 - u0).max()) <= 1e-5 * float(abs(u0).max())
    s.close()


TAIL, FINEST = 4096, 1 << 20  # cells: the levels below are the tail's; what boxes of 4096 cells hold


@pytest.mark.gpu
@pytest.mark.parametrize("poisson,dims,perdir", [
    ("refined", (256, 200), ()), ("refined", (200, 136), (1, 2)), ("refined", (2048, 16), (2,)),
    ("refined", (16, 2048), (1,)), ("refined", (64, 64, 64), ()), ("refined", (120, 88, 72), (1, 2)),
    ("refined", (100, 60, 84), (3,)), ("refined", (512, 16, 16), (1, 2, 3)), ("refined", (16, 256, 32), ()),
    ("refined", (160, 160, 96), (2,)), ("refined", (240, 208, 200), (1,)), ("refined", (256, 256, 248), (3,)),
    ("reference", (64, 64), (1, 2)), ("reference", (256, 200), ()), ("reference", (1000, 24), (2,)),
    ("reference", (512, 512), ()), ("reference", (1024, 640), (1,)), ("reference", (48, 32, 40), ()),
    ("reference", (100, 60, 84), (1, 3)), ("reference", (64, 64, 64), ()), ("reference", (96, 96, 96), (2,)),
    ("reference", (128, 128, 128), ()),
])
def test_every_level_above_the_tail_takes_one_launch(poisson, dims, perdir):
    """The grids of test_coarse_cg.py: the levels above the tail (and the finest
    in the default solver), up to 2M cells in 3D and 1M otherwise, are solved in
    one launch each in every V-cycle, the coarsest of them on one XCD (the XCDs
    were read on the device), and none gives up."""
    say("levels in one launch", poisson, dims, perdir)
    kw = dict(poisson_tol=1e-12, poisson_itmx=3) if poisson == "reference" else {}
    s, u = box(dims, perdir, poisson=poisson, **kw)
    _, _, st = project(s, u)
    o = info(s)
    want = 0
    for l in range(s._lib.ia_mg_levels(s._ctx, 0, None)):
        cells = int(np.prod([n >> l for n in dims]))
        big = 2 * FINEST if poisson == "refined" and len(dims) == 3 else FINEST
        if cells <= big and (cells > TAIL or l == 0) and l >= (poisson == "refined"):
            want |= 1 << l
    assert o.levels == want and want
    nl, nn = bin(want).count("1"), bin(o.near_levels).count("1")
    assert o.near_levels & (1 << (want.bit_length() - 1))
    assert o.solves in (st.iters * nl, (st.iters + 1) * nl)  # the flexible CG queues one V-cycle ahead
    assert o.solves_near == st.iters * nn
    assert o.given_up == 0 and o.rest == 0
    s.close()


@pytest.mark.gpu
def test_launches_per_iteration_are_none_of_these(monkeypatch):
    say("no level in one launch with IA_CG1_NB")
    monkeypatch.setenv("IA_CG1_NB", "256")
    s, u = box((192, 136), poisson="refined")
    project(s, u)
    o = info(s)
    assert o.levels == 0 and o.solves == 0 and o.solves_near == 0 and o.given_up == 0
    s.close()


WIDE = dict(dims=(256, 256, 248), poisson="refined")   # a level of one workgroup per CU
FLAT = dict(dims=(1024, 640), poisson="reference", poisson_tol=1e-12, poisson_itmx=40)  # 160 workgroups on the finest level
NEAR = dict(dims=(192, 136), poisson="refined")        # on one XCD


@pytest.mark.gpu
@pytest.mark.parametrize("kinds", [(WIDE, WIDE), (FLAT, FLAT), (WIDE, NEAR, FLAT), (NEAR,) * 10])
def test_contexts_at_once(kinds):
    """Contexts that project at the same time from threads of their own: nobody
    gives up, and everyone's bits are those of its projection alone (the same
    launches, only later)."""
    say("one-launch solves of contexts at once", [k["dims"] for k in kinds])
    sims = [box(perdir=(), seed=3 + i, **k) for i, k in enumerate(kinds)]
    alone = [project(s, u)[:2] for s, u in sims]
    gate, wrong = threading.Barrier(len(sims)), []

    def work(i):
        s, u = sims[i]
        gate.wait()
        for _ in range(6):
            uk, pk, _ = project(s, u)
            if not ((uk == alone[i][0]).all() and (pk == alone[i][1]).all()):
                wrong.append(i)

    ts = [threading.Thread(target=work, args=(i,)) for i in range(len(sims))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    got = [info(s) for s, _ in sims]
    assert all(o.given_up == 0 and o.solves > 0 for o in got), [o.given_up for o in got]
    assert not wrong
    for s, _ in sims:
        s.close()
