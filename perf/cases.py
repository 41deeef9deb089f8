"""The workloads that this package's speed is measured on.

Each case is one thing that a program built on the package does again and
again, called through the package's own entry points on the GPU:

- "step": a simulation (re)started from a given state and stepped, `sim_step_`;
  its arrays are the program's own device buffers, adopted with
  `ia_attach_field`.  Solver, element type, plug-ins, walls or periodic axes as
  the case says;
- "project": one pressure projection for a program that drives the step itself
  (`ia_update_L`, `ia_mg_update`, `ia_project`);
- "advect": `advect_`, interface transport by a given velocity, FP64 or FP32;
- "redistance": `LevelSet` + `redistaning_` of an interface field.

Sides are multiples of 4 (MultiLevelPoisson coarsens a grid at least twice).
"""
import math
import os
import random

import numpy as np
import torch

from __graft_entry__ import load_package

ia = load_package()
DEV = "cuda"
EPS = {"f32": 2.0 ** -23, "f64": 2.0 ** -52}


def listed():
    return [
        # pure interface transport on a small 2D grid: a few launches of a few microseconds each
        dict(name="advect_2d_128_f64", kind="advect", nx=128, ny=128, nz=0, dtype="f64", periodic="xy", nb=1),
        # the same in 3D between walls, no side a power of two, partly filled tiles
        dict(name="advect_3d_200x132x148_f32", kind="advect", nx=200, ny=132, nz=148, dtype="f32", periodic="", nb=12),
        # the periodic droplet of the smallest whole-step runs, default solver
        dict(name="step_2d_64_f64_periodic", kind="step", nx=64, ny=64, nz=0, dtype="f64", periodic="xy", nb=1,
             poisson="reference", steps=2, pool=False, eta=0.0, scheme="WH", limiter="Koren", amp=0.9),
        # the 2D two-phase box from rest: a few V-cycles a solve at first, the default solver's limit of 200 later
        dict(name="step_2d_256_f32_box", kind="step", nx=256, ny=256, nz=0, dtype="f32", periodic="", nb=1,
             poisson="reference", steps=12, pool=True, eta=0.0, scheme="WH", limiter="Koren", amp=0.0),
        # a wider 2D box with the solver to a relative residual
        dict(name="step_2d_384x256_f32_refined", kind="step", nx=384, ny=256, nz=0, dtype="f32", periodic="", nb=3,
             poisson="refined", steps=1, pool=True, eta=0.0, scheme="WH", limiter="Koren"),
        # 3D FP64 with surface tension and other plug-ins, one periodic axis, default solver
        dict(name="step_3d_48_f64_tension", kind="step", nx=48, ny=48, nz=48, dtype="f64", periodic="x", nb=2,
             poisson="reference", steps=1, pool=False, eta=0.5, scheme="MYC", limiter="minmod"),
        # a small 3D pool: coarse levels and launches dominate
        dict(name="step_3d_64_f32_pool", kind="step", nx=64, ny=64, nz=64, dtype="f32", periodic="", nb=8,
             poisson="refined", steps=2, pool=True, eta=0.0, scheme="WH", limiter="Koren"),
        # the benchmark's pool of bubbles, 256^3
        dict(name="step_3d_256_f32_pool", kind="step", nx=256, ny=256, nz=256, dtype="f32", periodic="", nb=32,
             poisson="refined", steps=2, pool=True, eta=0.0, scheme="WH", limiter="Koren"),
        # the largest configuration, a 512^3 slab with 256 bubbles
        dict(name="step_3d_512_f32_slab", kind="step", nx=512, ny=512, nz=512, dtype="f32", periodic="", nb=256,
             poisson="refined", steps=1, pool=True, eta=0.0, scheme="WH", limiter="Koren"),
        # a step whose solves start from the trained network's correction
        dict(name="step_3d_128_f32_learned", kind="step", nx=128, ny=128, nz=128, dtype="f32", periodic="", nb=16,
             poisson="learned", steps=1, pool=True, eta=0.0, scheme="WH", limiter="Koren"),
        # one projection on a box of unequal sides that halve to odd ones, periodic in x and y
        dict(name="project_3d_120x88x72_f32", kind="project", nx=120, ny=88, nz=72, dtype="f32", periodic="xy", nb=6,
             poisson="refined"),
        # reinitialisation of the benchmark-sized interface field
        dict(name="redistance_3d_256_f32", kind="redistance", nx=256, ny=256, nz=256, dtype="f32", periodic="", nb=32,
             d=2.0, dtau=0.5),
    ]


def _side(rng, lo, hi):
    """A multiple of 4 in [lo, hi], spread over the logarithm."""
    return max(lo, min(hi, 4 * round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / 4)))


def draw(rng):
    kind = rng.choice(["advect", "step", "step", "step", "project", "redistance"])
    two = rng.random() < (0.4 if kind in ("step", "advect") else 0.0)
    per = "".join(a for a in ("xy" if two else "xyz") if rng.random() < 0.3)
    c = dict(kind=kind, nz=0, periodic=per, dtype="f32", nb=rng.randint(1, 3) if two else rng.randint(2, 12))
    if kind == "advect":
        c.update(nx=_side(rng, 32, 1024 if two else 256), ny=_side(rng, 32, 1024 if two else 256),
                 nz=0 if two else _side(rng, 32, 256), dtype=rng.choice(["f32", "f64"]))
    elif kind == "redistance":
        c.update(nx=_side(rng, 32, 320), ny=_side(rng, 32, 320), nz=_side(rng, 32, 320), d=rng.choice([1.0, 2.0, 3.0]),
                 dtau=0.5)
    elif kind == "project":
        c.update(nx=_side(rng, 48, 288), ny=_side(rng, 48, 288), nz=_side(rng, 48, 288), poisson="refined")
    elif two:
        mode = rng.choice(["reference", "refined"])
        c.update(nx=_side(rng, 48, 512), ny=_side(rng, 48, 512), poisson=mode, steps=rng.randint(1, 3), pool="y" not in per, eta=0.0,
                 scheme=rng.choice(["WH", "WH", "Column", "WY"]), limiter=rng.choice(["Koren", "Koren", "superbee"]),
                 amp=rng.choice([0.0, 0.2, 0.7]))
    else:
        c.update(nx=_side(rng, 48, 288), ny=_side(rng, 48, 288), nz=_side(rng, 48, 288), poisson="refined", steps=1,
                 pool="z" not in per, eta=0.0, scheme=rng.choice(["WH", "WH", "MYC"]),
                 limiter=rng.choice(["Koren", "Koren", "minmod"]))
    return c


# --------------------------------------------------------------------------- inputs
def _dims(c):
    return (c["nx"], c["ny"]) + ((c["nz"],) if c["nz"] else ())


def _axes(dims, shift=0.0):
    """Cell-centre coordinates (ghosts included) per axis, as broadcastable tensors; arrays are [z, y, x]."""
    D = len(dims)
    out = []
    for a, n in enumerate(dims):
        x = torch.arange(n + 2, dtype=torch.float64, device=DEV) - 0.5 + shift
        out.append(x.reshape([-1 if D - 1 - k == a else 1 for k in range(D)]))
    return out


def _sl(D, a, s):
    """Index `s` along axis a (0 = x) of a [.., y, x] array."""
    ix = [slice(None)] * D
    ix[D - 1 - a] = s
    return tuple(ix)


def _bc_scalar(q, per):
    D = q.dim()
    for a in range(D):
        lo, hi = (-2, 1) if per[a] else (1, -2)
        q[_sl(D, a, 0)] = q[_sl(D, a, lo)]
        q[_sl(D, a, -1)] = q[_sl(D, a, hi)]
    return q


def _fraction(c, rng):
    """Volume fraction of liquid: a pool under a free surface (or all liquid) with gas spheres that do not touch,
    or liquid drops in gas; one cell wide at the interface, as a cell fraction is."""
    dims, D = _dims(c), len(_dims(c))
    per = [a in c["periodic"] for a in "xyz"[:D]]
    X = _axes(dims)
    H, m = dims[-1], min(dims)
    pool = c.get("pool", True) and not per[-1]
    top = H * rng.uniform(0.6, 0.72)
    got, tries = [], 0
    while len(got) < c["nb"] and tries < 20000:
        tries += 1
        r = m * (rng.uniform(0.12, 0.2) if c["nb"] == 1 else rng.uniform(0.04, 0.08) if c["nb"] < 100
                 else rng.uniform(0.02, 0.05))
        x = [rng.uniform(r + 2, n - r - 2) for n in dims]
        if pool:
            x[-1] = rng.uniform(r + 2, max(r + 2.5, top - r - 2))
        if all(math.dist(x, y) > r + s + 2 for y, s in got):
            got.append((x, r))
    if pool:
        wave = sum(0.02 * H * torch.cos(math.pi * rng.randint(1, 2) * (2 if per[a] else 1) * X[a] / dims[a])
                   for a in range(D - 1))
        phi = (X[-1] - top - wave).expand([n + 2 for n in reversed(dims)]).to(torch.float32).clone()
    else:
        phi = torch.full([n + 2 for n in reversed(dims)], 1e3, dtype=torch.float32, device=DEV)
    for x, r in got:
        lo = [max(0, int(q - r - 4)) for q in x]
        hi = [min(n + 2, int(q + r + 6)) for q, n in zip(x, dims)]
        ix = tuple(slice(lo[a], hi[a]) for a in reversed(range(D)))
        d2 = 0
        for a in range(D):
            d2 = d2 + (X[a][_sl(D, a, slice(lo[a], hi[a]))] - x[a]) ** 2
        s = (torch.sqrt(d2) - r).to(torch.float32)
        phi[ix] = torch.maximum(phi[ix], -s) if pool else torch.minimum(phi[ix], s)
    f = (0.5 - phi).clamp_(0, 1).to(torch.float64 if c["dtype"] == "f64" else torch.float32)
    return _bc_scalar(f, per)


def _mode(x, n, periodic, k, ph):
    return torch.cos(2 * math.pi * k * x / n + ph) if periodic else torch.sin(math.pi * k * x / n)


def _velocity(c, rng, amp):
    """A staggered velocity whose discrete divergence is zero, from stream functions of a few modes, zero through
    walls, with max |u| = amp; ghosts as the package's BC! leaves them."""
    dims, D = _dims(c), len(_dims(c))
    per = [a in c["periodic"] for a in "xyz"[:D]]
    shape = [n + 2 for n in reversed(dims)]
    u = torch.zeros([D] + shape, dtype=torch.float64 if c["dtype"] == "f64" else torch.float32, device=DEV)
    X = _axes(dims)
    for a, b in ([(0, 1)] if D == 2 else [(0, 1), (1, 2), (2, 0)]):
        for _ in range(2):
            ka, kb, kc = rng.randint(1, 3), rng.randint(1, 3), rng.randint(0, 2)
            pa, pb, s = rng.uniform(0, 6), rng.uniform(0, 6), rng.uniform(0.4, 1) * rng.choice([-1, 1])
            w = s * math.sqrt(dims[a] * dims[b])
            lo = [x - 0.5 for x in X]  # lower corner of every cell
            A0, A1 = _mode(lo[a], dims[a], per[a], ka, pa), _mode(lo[a] + 1, dims[a], per[a], ka, pa)
            B0, B1 = _mode(lo[b], dims[b], per[b], kb, pb), _mode(lo[b] + 1, dims[b], per[b], kb, pb)
            if D == 3:
                q = 3 - a - b
                w = w * torch.cos(math.pi * kc * (2 if per[q] else 1) * X[q] / dims[q])
            u[a] += (w * A0 * (B1 - B0)).to(u.dtype)
            u[b] -= (w * B0 * (A1 - A0)).to(u.dtype)
    u *= amp / float(u.abs().max())  # amp 0: from rest
    for i in range(D):
        for a in range(D):
            v = u[i]
            if per[a]:
                v[_sl(D, a, 0)] = v[_sl(D, a, -2)]
                v[_sl(D, a, -1)] = v[_sl(D, a, 1)]
            elif a == i:
                for s in (0, 1, -1):
                    v[_sl(D, a, s)] = 0
            else:
                v[_sl(D, a, 0)] = v[_sl(D, a, 1)]
                v[_sl(D, a, -1)] = v[_sl(D, a, -2)]
    return u


def _dt(c):
    return 0.5 if c["kind"] == "project" else 0.4


def _inputs(c, seed):
    rng = random.Random(int(seed))
    f = _fraction(c, rng)
    amp = {"advect": 0.8, "project": 0.3}.get(c["kind"], c.get("amp", 0.2))
    u = _velocity(c, rng, amp) if c["kind"] != "redistance" else None
    if c["kind"] == "project":  # what a viscous step adds: a divergence near the interface
        D = f.dim()
        for i in range(D):
            g = torch.zeros_like(f)
            g[_sl(D, i, slice(2, -1))] = 0.1 * (f[_sl(D, i, slice(2, -1))] - f[_sl(D, i, slice(1, -2))])
            u[i] += g
    return f, u


def prepare(case, seed):
    c = case
    dims, D = _dims(c), len(_dims(c))
    T = np.float64 if c["dtype"] == "f64" else np.float32
    L = float(dims[-1])
    kw = dict(T=T, perdir=tuple(a + 1 for a in range(D) if "xyz"[a] in c["periodic"]))
    if c["kind"] in ("step", "project"):
        kw.update(λρ=1e-3 if c.get("pool", True) else 0.1, λμ=1e-2, ν=L / 1e4, poisson=c["poisson"],
                  poisson_max_outer=200, λ=c.get("limiter", "Koren"), normalScheme=c.get("scheme", "WH"))
        if c.get("pool", True):
            kw["g"] = (0.0,) * (D - 1) + (-1.0 / L,)
        if c.get("eta"):
            kw["η"] = c["eta"]
    sim = ia.TwoPhaseSimulation(dims, (0.0,) * D, L, **kw)
    if c.get("poisson") == "learned":
        sim.learned_weights = np.fromfile(os.path.join(os.path.dirname(ia.__file__), "learned_pool256.f32"), "<f4")
    f, u = _inputs(c, seed)
    own = {"f": f.clone(), "f0": f.clone()}
    if u is not None:
        own.update(u=u.clone(), u0=u.clone())
    if c["kind"] in ("step", "project"):
        own["p"] = torch.zeros_like(f)
    torch.cuda.synchronize()
    for k, t in own.items():
        sim._call("ia_attach_field", ia.FIELD[k], ia.C.c_void_p(t.data_ptr()), t.numel() * t.element_size())
    st = dict(case=c, sim=sim, own=own)
    if c["kind"] == "step":
        sim.flow.Δt[-1] = min(sim.flow.Δt[-1], sim.T.type(sim.MPCFL()))
        st.update(Δt=list(sim.flow.Δt))
    if c["kind"] in ("step", "project"):
        st.update(start=dict(f=f, f0=f, u=u, u0=u, p=torch.zeros_like(f)))
    sim._call("ia_synchronize")
    return st


def _put(sim, name, t):
    sim._call("ia_set_field", ia.FIELD[name], ia.C.c_void_p(t.data_ptr()), t.numel() * t.element_size())


def run(state):
    c, sim, own = state["case"], state["sim"], state["own"]
    if c["kind"] == "advect":
        ia.advect_(sim, dt=_dt(c))
        return {"f": own["f"]}
    if c["kind"] == "redistance":
        ia.redistaning_(ia.LevelSet(sim), d=c["d"], dτ=c["dtau"], perdir=sim.perdir)
        return {"phi": own["f0"]}
    start = state["start"]
    if c["kind"] == "project":
        for k in ("u", "p"):
            _put(sim, k, start[k])
        sim._call("ia_update_L", 0)
        sim._call("ia_mg_update")
        sim._call("ia_project", _dt(c), None)
        sim._call("ia_synchronize")  # the program's own kernels read u next
        return {"u": own["u"], "p": own["p"]}
    for k, t in start.items():
        _put(sim, k, t)
    sim.flow.Δt[:] = state["Δt"]
    for _ in range(c["steps"]):
        ia.sim_step_(sim)
    return {"f": own["f"], "u": own["u"], "p": own["p"], "dt": float(sim.flow.Δt[-1])}


def work(case):
    dims, D = _dims(case), len(_dims(case))
    n = math.prod(dims) * (8 if case["dtype"] == "f64" else 4)
    # fields read once + fields written once, per pass
    arrays = {"advect": (1 + 2 * D) + 1, "redistance": 1 + 1, "project": (1 + D + 1) + (D + 1),
              "step": ((1 + D + 1) + (2 + 2 * D + 1)) * case.get("steps", 1)}[case["kind"]]
    return {"bytes": float(n * arrays), "flops": 0.0}


# --------------------------------------------------------------------------- the same in 64 bits
def _sh(q, a, k):
    """q[I + k e_a], the outermost layer kept where there is none."""
    return torch.roll(q, -k, q.dim() - 1 - a)


def _sum3(q, s):
    return q + _sh(q, s, -1) + _sh(q, s, 1)


def _pick(vals, k):
    out = vals[0].clone()
    for a in range(1, len(vals)):
        out = torch.where(k == a, vals[a], out)
    return out


def _argabsmax(n):
    best, at = torch.zeros_like(n[0]), torch.zeros_like(n[0], dtype=torch.long)
    for a, v in enumerate(n):
        at = torch.where(v * v > best, a, at)
        best = torch.maximum(best, v * v)
    return at


def _normal_wh(f):
    D = f.dim()
    n = [_sh(f, a, -1) - _sh(f, a, 1) for a in range(D)]
    dom = _argabsmax(n)
    h = [_sum3(f, s) for s in range(D)]
    for a in range(D):
        side = _pick([(_sh(h[s], a, -1) - _sh(h[s], a, 1)) / 2 for s in range(D)], dom)
        n[a] = torch.where(dom == a, torch.where(n[a] < 0, -1.0, 1.0).to(f.dtype), side)
    im = _argabsmax(n)
    nim = _pick(n, im)
    an = torch.where(nim == 0, torch.ones_like(nim), nim.abs())
    n = [v / an for v in n]
    for a in range(D):
        slope, up = n[a].abs(), ~torch.signbit(n[a])
        hm, hp = _pick([_sh(h[s], a, -1) for s in range(D)], im), _pick([_sh(h[s], a, 1) for s in range(D)], im)
        hl, hr = torch.where(up, hm, hp), torch.where(up, hp, hm)
        sh = hl + _pick(h, im) + hr
        s45 = 4.5 * slope
        mn = torch.minimum(s45, 1 / (2 * slope))
        wm, wp = _pick([_sh(h[a], s, -1) for s in range(D)], im), _pick([_sh(h[a], s, 1) for s in range(D)], im)
        wb, wt = torch.where(torch.signbit(nim), wp, wm), torch.where(torch.signbit(nim), wm, wp)
        sg = torch.where(up, 1.0, -1.0).to(f.dtype)
        low = (sh < s45) & (wb > mn) & (im != a)
        high = (sh > 9 - s45) & (wt < 3 - mn) & (im != a)
        v = torch.where(low, ((hl - 0.5) / (wb - 0.5)).abs() * sg, n[a])
        n[a] = torch.where(high, ((2.5 - hr) / (2.5 - wt)).abs() * sg, v)
    return n


def _sorted_abs(n):
    m, _ = torch.sort(torch.stack([v.abs() for v in n]), dim=0)
    t = m.sum(0)
    return [v / t for v in m], t


def _volume(n, al):
    """The part of the unit cell under the plane n·x = al."""
    m, t = _sorted_abs(n)
    a = (al - sum(v.clamp(max=0) for v in n)) / t
    b = torch.minimum(a, 1 - a)
    if len(n) == 2:
        m1, m2 = m
        v = torch.where(b < m1, b * b / (2 * m1 * m2), (b - m1 / 2) / m2)
    else:
        m1, m2, m3 = m
        m12, p = m1 + m2, 6 * m1 * m2 * m3
        v1 = torch.where(m2 == 0, torch.ones_like(m1), m1 / m2) * m1 / (6 * m3)
        c3 = b * b * (3 * m12 - b) + m1 * m1 * (m1 - 3 * b) + m2 * m2 * (m2 - 3 * b)
        c4 = b * b * (3 - 2 * b) + m1 * m1 * (m1 - 3 * b) + m2 * m2 * (m2 - 3 * b) + m3 * m3 * (m3 - 3 * b)
        v = torch.where(m3 < m12, c4 / p, (2 * b - m12) / (2 * m3))
        v = torch.where(b < torch.minimum(m3, m12), c3 / p, v)
        v = torch.where(b < m2, b * (b - m1) / (2 * m2 * m3) + v1, v)
        v = torch.where(b < m1, b ** 3 / p, v)
    v = torch.where(a < 0.5, v, 1 - v)
    return torch.where((a <= 0) | (a >= 1) | (a == 0.5), a.clamp(0, 1), v)


def _intercept(n, f):
    """al with _volume(n, al) = f: the volume is monotonic in al, so 60 halvings, then two Newton-like secants."""
    lo = sum(v.clamp(max=0) for v in n)
    hi = sum(v.clamp(min=0) for v in n)
    for _ in range(60):
        mid = (lo + hi) / 2
        small = _volume(n, mid) < f
        lo, hi = torch.where(small, mid, lo), torch.where(small, hi, mid)
    return (lo + hi) / 2


def _exact_advect(c, seed, first=3):
    f, u = _inputs(c, seed)
    dims, D, T = _dims(c), f.dim(), c["dtype"]
    f, u = f.double(), u.double()
    per = [a in c["periodic"] for a in "xyz"[:D]]
    dt, tol = _dt(c), 10 * EPS[T]
    dt = float(np.float32(dt)) if T == "f32" else dt
    inner = tuple(slice(1, -1) for _ in range(D))
    cb = (f >= 0.5).double()
    for i in range(1, D + 1):
        d = (1 + i) % D  # a simulation before its first step: length(Δt) = 1
        dl = dt * u[d]
        mixed = (f > 0) & (f < 1)
        edge = torch.ones_like(mixed)
        edge[inner] = False
        at = torch.nonzero((mixed & ~edge).reshape(-1)).reshape(-1)
        n = [v.reshape(-1)[at] for v in _normal_wh(f)]
        al = _intercept(n, f.reshape(-1)[at])
        flux = {}
        for up in (True, False):  # swept out of the cell through its upper face (dl > 0) or its lower one (dl < 0)
            dd = (_sh(dl, d, 1) if up else dl).reshape(-1)[at]
            nc = [v * dd.abs() if a == d else v for a, v in enumerate(n)]
            part = torch.nan_to_num(_volume(nc, al - n[d] * (1 - dd) if up else al))
            q = f.clone().reshape(-1)
            q[at] = part
            q = q.reshape(f.shape)
            if per[d]:
                q[_sl(D, d, 0)] = q[_sl(D, d, -2)]
                q[_sl(D, d, -1)] = q[_sl(D, d, 1)]
            flux[up] = q
        face = torch.where(dl > 0, _sh(flux[True], d, -1), flux[False]) * dl
        new = f + (face - _sh(face, d, 1)) + cb * (_sh(u[d], d, 1) - u[d]) * dt
        new = torch.where(new < tol, 0.0, torch.where(new > 1 - tol, 1.0, new))
        f = f.clone()
        f[inner] = new[inner]
        f = _bc_scalar(f, per)
    return {"f": f}


def _exact_redistance(c, seed):
    f, _ = _inputs(c, seed)
    D = f.dim()
    per = [a in c["periodic"] for a in "xyz"[:D]]
    phi = 2 * f.double() - 1
    ini, sgn = phi.clone(), torch.sign(phi)
    mm = lambda a, b: torch.where(a.abs() <= b.abs(), a, b)  # noqa: E731

    def rate(q):
        g2 = torch.zeros_like(q)
        for a in range(D):
            b, d = _sh(q, a, -1), _sh(q, a, 1)
            aa, ee = _sh(q, a, -2), _sh(q, a, 2)
            s1, s2 = _sl(D, a, 1), _sl(D, a, -2)
            aa[s1] = q[_sl(D, a, -3)] if per[a] else b[s1]
            ee[s2] = q[_sl(D, a, 2)] if per[a] else d[s2]
            o = d + b - 2 * q
            R = d - q - mm(ee + q - 2 * d, o) / 2
            Lf = q - b + mm(o, q + aa - 2 * b) / 2
            wR, wL = R * sgn, Lf * sgn
            g2 += torch.where((wR < 0) & (wR + wL < 0), R * R, torch.where((wL > 0) & (wR + wL > 0), Lf * Lf, 0.0))
        return ini * (1 - torch.sqrt(g2))

    for _ in range(round(c["d"] / c["dtau"])):
        old = phi
        for al in (0.0, 3.0 / 4, 1.0 / 3):
            new = phi.clone()
            i = tuple(slice(1, -1) for _ in range(D))
            new[i] = (al * old + (1 - al) * (phi + c["dtau"] * rate(phi)))[i]
            phi = _bc_scalar(new, per)
    return {"phi": phi}


def _exact_project(c, seed):
    """u - L ∇x with ∇·(L ∇x) = ∇·u, by conjugate gradients to round-off."""
    f, u = _inputs(c, seed)
    dims, D = _dims(c), f.dim()
    per = [a in c["periodic"] for a in "xyz"[:D]]
    f, u = f.double(), u.double()
    i = tuple(slice(1, -1) for _ in range(D))
    lam = 1e-3
    Lc = []
    for a in range(D):
        q = 1 / (lam + (1 - lam) * (f + _sh(f, a, -1)) / 2)[i]
        if not per[a]:
            q[_sl(D, a, 0)] = 0
        Lc.append(q)
        if not per[a]:
            assert float(u[a][i][_sl(D, a, 0)].abs().max()) == 0
    # on the interior, a roll is the periodic image; across a wall the coefficient is 0
    A = lambda x: sum(_sh(Lc[a] * (x - _sh(x, a, -1)), a, 1) - Lc[a] * (x - _sh(x, a, -1)) for a in range(D))  # noqa: E731
    ui = [u[a][i].clone() for a in range(D)]
    z = sum((_sh(u[a], a, 1) - u[a])[i] for a in range(D))
    z = z - z.mean()
    diag = -sum(Lc[a] + _sh(Lc[a], a, 1) for a in range(D))
    x, r = torch.zeros_like(z), z.clone()
    y = r / diag
    p, rho, z2 = y.clone(), (r * y).sum(), float(z.norm())
    for k in range(20000):
        q = A(p)
        al = rho / (p * q).sum()
        x += al * p
        r -= al * q
        if k % 100 == 99 and float(r.norm()) <= 1e-12 * z2:
            break
        y = r / diag
        rho, old = (r * y).sum(), rho
        p = y + (rho / old) * p
    for a in range(D):
        u[a][i] = ui[a] - Lc[a] * (x - _sh(x, a, -1))
    for b in range(D):
        for a in range(D):
            v = u[b]
            if per[a]:
                v[_sl(D, a, 0)] = v[_sl(D, a, -2)]
                v[_sl(D, a, -1)] = v[_sl(D, a, 1)]
            elif a != b:
                v[_sl(D, a, 0)] = v[_sl(D, a, 1)]
                v[_sl(D, a, -1)] = v[_sl(D, a, -2)]
            else:
                for s in (0, 1, -1):
                    v[_sl(D, a, s)] = 0
    return {"u": u, "p": None}  # p is defined up to a constant


def exact(case, seed):
    if case["kind"] == "advect":
        return _exact_advect(case, seed)
    if case["kind"] == "redistance":
        return _exact_redistance(case, seed)
    if case["kind"] == "project":
        return _exact_project(case, seed)
    # a step holds two pressure solves that stop at a tolerance between its sweeps: solving both to round-off with
    # plain tensor operations takes minutes at these sizes
    return None
