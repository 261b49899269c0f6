"""Workloads that stand for what a program does with this package, each as one
pass through its public entry points.

listed() gives the fixed workloads, draw(rng) another one of the same ranges;
prepare(case, seed) makes what a program holds before the call, run(state) is
the call, work(case) the bytes and operations it cannot do without, and
exact(case, seed) its results in 64 bits from plain torch.

Kinds of work:
  gas      the split MUSCL-Hancock step loop on one grid (SplitSolver.simulate);
           a pass goes on from the state that the last one left
  bubble   the two-material ghost-fluid loop (MultimaterialSimulator.simulate_mm)
           from a given initial state
  batch    many uneven grids advanced together (Batch.step, Batch.finish)
  adjoint  a checkpointed run forward and its gradient (Adjoint.forward, .backward)

Initial states are Riemann data (two or four constant states) with smooth
perturbations of a few percent on top, so that every cell of a grid takes part
from the first step on, as it does in a run that has gone on for a while.
"""
from __future__ import annotations

import math
import random

import torch

CFL = 0.9
GAMMA = 1.4
PAD = 4  # cells a split sweep reads on either side


def listed():
    def gas(name, nx, ny, steps, **kw):
        c = dict(name=name, kind="gas", nx=nx, ny=ny, steps=steps, dtype="f64", layout="aos",
                 numerics="exact", flux="hllc", limiter="vanleer", form="cons", bc="transmissive")
        return {**c, **kw}

    return [
        # The shock tubes of the textbook tests: one line of a hundred cells,
        # nothing but latency.
        gas("tube_100", 100, 0, 200),
        # The reference's own one-dimensional configuration, part of its run.
        gas("tube_4096", 4096, 0, 400),
        # A long line of odd length in the fast numerics, planes per component.
        gas("tube_150001_fast", 150001, 0, 64, layout="soa", numerics="fast", flux="force"),
        # The smallest planes: tests, tuning of a setup, coarse sweeps of parameters.
        gas("plane_64", 64, 64, 64),
        # An ordinary plane of ragged size with the other choice of every option.
        gas("plane_509x317_force", 509, 317, 16, layout="soa", flux="force", limiter="superbee",
            form="prim", bc="reflective"),
        # Single precision on an ordinary plane.
        gas("plane_1024_f32", 1024, 1024, 16, dtype="f32", layout="soa"),
        # A large plane in the defaults of the solver: the reference's bits and its layout.
        gas("plane_2048", 2048, 2048, 4),
        # The headline workload of bench.py: 4096 x 4096, fast numerics.
        gas("plane_4096_fast", 4096, 4096, 4, layout="soa", numerics="fast"),
        # A coarse shock-bubble run in the defaults: reinitialised every step.
        dict(name="bubble_384x192", kind="bubble", nx=384, ny=192, steps=6, numerics="exact",
             layout="aos", reinit=1),
        # The shock-bubble workload of bench.py.
        dict(name="bubble_2048x1024_fast", kind="bubble", nx=2048, ny=1024, steps=5,
             numerics="fast", layout="soa", reinit=5),
        # A parameter study: lines of 256 to 65536 cells and planes of 64 to 1024 a side.
        dict(name="batch_48", kind="batch", lines=32, planes=16, longest=65536, widest=1024,
             steps=8, dtype="f64", numerics="exact", layout="soa"),
        # Gradient of a misfit with respect to the initial state and gamma.
        dict(name="adjoint_512", kind="adjoint", nx=512, ny=512, steps=20, every=10, flux="hllc",
             form="cons", layout="soa"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["tube", "tube", "plane", "plane", "plane", "bubble", "batch", "adjoint"])
    layout = rng.choice(["aos", "soa"])
    numerics = rng.choice(["exact", "exact", "fast"])
    if kind in ("tube", "plane"):
        if kind == "tube":
            nx, ny = _log_int(rng, 64, 200000), 0
            steps = _log_int(rng, 32, 400)
        else:
            nx, ny = _log_int(rng, 48, 4096), _log_int(rng, 48, 4096)
            # the dearest options at this many cells and steps cost what the
            # largest listed case does
            steps = max(2, min(_log_int(rng, 4, 64), 3 * 4096 * 4096 // (nx * ny)))
        form = rng.choice(["cons", "cons", "prim"])
        return dict(kind="gas", nx=nx, ny=ny, steps=steps, dtype=rng.choice(["f64", "f64", "f32"]),
                    layout=layout, numerics=numerics, flux=rng.choice(["hllc", "hllc", "force"]),
                    limiter=rng.choice(["vanleer", "vanleer", "superbee"]), form=form,
                    bc=rng.choice(["transmissive", "reflective", "periodic"]))
    if kind == "bubble":
        ny = _log_int(rng, 128, 900)
        nx = int(ny * rng.uniform(1.5, 2.2))
        return dict(kind="bubble", nx=nx, ny=ny, steps=rng.randint(2, 6), numerics=numerics,
                    layout=layout, reinit=rng.choice([1, 2, 5]))
    if kind == "batch":
        return dict(kind="batch", lines=rng.randint(8, 36), planes=rng.randint(4, 20),
                    longest=_log_int(rng, 4096, 65536), widest=_log_int(rng, 256, 1024),
                    steps=rng.randint(4, 10), dtype=rng.choice(["f64", "f64", "f32"]),
                    numerics=numerics, layout=layout)
    return dict(kind="adjoint", nx=_log_int(rng, 64, 600), ny=_log_int(rng, 64, 600),
                steps=rng.randint(6, 20), every=rng.randint(4, 20),
                flux=rng.choice(["hllc", "force"]), form=rng.choice(["cons", "prim"]),
                layout=layout)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _rng(seed, salt):
    return random.Random(int(seed) * 1000003 + salt)


def _modes(r, axes, count=8):
    """A smooth field of mean 0 and amplitude about 1: random sine waves over the grid."""
    f = 0.0
    for _ in range(count):
        phase = 2 * math.pi * r.random()
        for x in axes:
            phase = phase + 2 * math.pi * r.randint(1, 8) * x
        f = f + torch.sin(phase)
    return f / math.sqrt(count)


def _axes(shape):
    """Cell-centre coordinates in [0, 1] per dimension, x first, as broadcastable tensors."""
    n = len(shape)
    out = []
    for d in range(n):
        x = (torch.arange(shape[n - 1 - d], dtype=torch.float64, device="cuda") + 0.5)
        x = x / shape[n - 1 - d]
        out.append(x.view([-1 if a == n - 1 - d else 1 for a in range(n)]))
    return out


def _cons(W, gamma):
    """Conservative planes [rho, E, m...] of primitive ones [rho, p, v...]."""
    rho, p, v = W[0], W[1], W[2:]
    E = p / (gamma - 1.0) + 0.5 * rho * sum(a * a for a in v)
    return torch.stack([rho, E] + [rho * a for a in v])


def _riemann(r, shape, gamma):
    """Conservative planes of two (1D) or four (2D) perturbed constant states."""
    axes, nd = _axes(shape), len(shape)
    at = [r.uniform(0.35, 0.65) for _ in range(nd)]
    W = [torch.zeros(shape, dtype=torch.float64, device="cuda") for _ in range(2 + nd)]
    for q in range(2 ** nd):
        inside = torch.ones(shape, dtype=torch.bool, device="cuda")
        for d in range(nd):
            inside = inside & ((axes[d] >= at[d]) == bool((q >> d) & 1))
        state = [math.exp(r.uniform(-0.7, 0.7)), math.exp(r.uniform(-0.9, 0.9))]
        state += [r.uniform(-0.4, 0.4) for _ in range(nd)]
        W = [torch.where(inside, torch.full_like(w, s), w) for w, s in zip(W, state)]
    W[0] = W[0] * (1.0 + 0.04 * _modes(r, axes))
    W[1] = W[1] * (1.0 + 0.04 * _modes(r, axes))
    for k in range(2, 2 + nd):
        W[k] = W[k] + 0.05 * _modes(r, axes)
    return _cons(torch.stack(W), gamma)


def _laid(U, layout, dtype="f64"):
    U = U.movedim(0, -1) if layout == "aos" else U
    return U.to(torch.float32 if dtype == "f32" else torch.float64).contiguous()


def _planes(U, layout):
    return (U.movedim(-1, 0) if layout == "aos" else U).double()


def _shape(case):
    return (case["ny"], case["nx"]) if case.get("ny") else (case["nx"],)


def _gas_input(case, seed):
    return _laid(_riemann(_rng(seed, 1), _shape(case), GAMMA), case["layout"], case["dtype"])


def _bubble_input(case, seed):
    """A planar shock in gas running onto a bubble of light gas: both materials'
    states over the whole grid, the bubble's signed distance and both gammas."""
    r = _rng(seed, 2)
    ny, nx = case["ny"], case["nx"]
    dh = 1.0 / ny
    g0, g1 = 1.4, 1.67
    radius = r.uniform(0.15, 0.25)
    cx, cy = nx * dh * r.uniform(0.45, 0.6), r.uniform(0.4, 0.6)
    mach = r.uniform(1.2, 2.5)
    m2 = mach * mach
    rho_s = (g0 + 1.0) * m2 / ((g0 - 1.0) * m2 + 2.0)
    p_s = (2.0 * g0 * m2 - (g0 - 1.0)) / (g0 + 1.0)
    u_s = mach * math.sqrt(g0) * (1.0 - 1.0 / rho_s)
    axes = _axes((ny, nx))
    x, y = axes[0] * nx * dh, axes[1]
    flat = torch.zeros((ny, nx), dtype=torch.float64, device="cuda")
    behind = (x + flat) < cx - radius - 0.05

    def pick(a, b):
        return torch.where(behind, torch.full_like(flat, a), torch.full_like(flat, b))
    W0 = torch.stack([pick(rho_s, 1.0) * (1.0 + 0.02 * _modes(r, axes)),
                      pick(p_s, 1.0) * (1.0 + 0.02 * _modes(r, axes)),
                      pick(u_s, 0.0) + 0.02 * _modes(r, axes), flat + 0.02 * _modes(r, axes)])
    W1 = torch.stack([0.14 * (1.0 + 0.02 * _modes(r, axes)), 1.0 + 0.02 * _modes(r, axes),
                      flat, flat])
    phi = torch.sqrt((x - cx) ** 2 + (y - cy) ** 2) - radius
    return _laid(_cons(W0, g0), case["layout"]), _laid(_cons(W1, g1), case["layout"]), phi, (g0, g1)


def _batch_sizes(case):
    """The grids of a batch: sizes spread over their logarithm, the same for every seed."""
    r = random.Random(17)
    shapes = [(_log_int(r, 256, case["longest"]),) for _ in range(case["lines"])]
    sides = [_log_int(r, 64, case["widest"]) for _ in range(case["planes"])]
    return shapes + [(n, n) for n in sides]


def _batch_input(case, seed):
    """Per problem (grid, gamma)."""
    out = []
    for i, shape in enumerate(_batch_sizes(case)):
        r = _rng(seed, 100 + i)
        gamma = r.uniform(1.2, 1.67)
        out.append((_laid(_riemann(r, shape, gamma), case["layout"], case["dtype"]), gamma))
    return out


def _adjoint_input(case, seed):
    """A smooth periodic flow and the density that its result is compared with."""
    r = _rng(seed, 3)
    axes = _axes((case["ny"], case["nx"]))
    W = torch.stack([1.0 + 0.1 * _modes(r, axes), 1.0 + 0.1 * _modes(r, axes),
                     0.5 + 0.1 * _modes(r, axes), 0.3 + 0.1 * _modes(r, axes)])
    return _laid(_cons(W, GAMMA), case["layout"]), 1.0 + 0.1 * _modes(r, axes)


# ---------------------------------------------------------------------------
# the framework's side
# ---------------------------------------------------------------------------

def _options(case, **kw):
    from fluidity_amd import euler as E
    from fluidity_amd import native as N
    bc = {"transmissive": N.FL_BC_TRANSMISSIVE, "reflective": N.FL_BC_REFLECTIVE,
          "periodic": N.FL_BC_PERIODIC}[kw.pop("bc", case.get("bc", "transmissive"))]
    return E.Scheme(
        limiter=N.FL_LIMITER_SUPERBEE if case.get("limiter") == "superbee" else N.FL_LIMITER_VAN_LEER,
        form=N.FL_FORM_PRIMITIVE if case.get("form") == "prim" else N.FL_FORM_CONSERVATIVE,
        flux=N.FL_FLUX_FORCE if case.get("flux") == "force" else N.FL_FLUX_HLLC,
        numerics=N.FL_NUMERICS_FAST if case.get("numerics") == "fast" else N.FL_NUMERICS_EXACT,
        bc=(bc, bc, bc), **kw)


def _layout(case):
    from fluidity_amd import native as N
    return N.FL_LAYOUT_AOS if case["layout"] == "aos" else N.FL_LAYOUT_SOA


def prepare(case, seed):
    s = {"case": case}
    if case["kind"] == "gas":
        from fluidity_amd import euler as E
        s["U"] = _gas_input(case, seed)
        s["work"] = torch.empty_like(s["U"])
        s["solver"] = E.SplitSolver(_options(case, gamma=GAMMA), layout=_layout(case))
    elif case["kind"] == "bubble":
        from fluidity_amd import levelset as L
        U0, U1, phi, gammas = _bubble_input(case, seed)
        s["initial"] = (U0, U1, -phi, phi)
        s["grids"] = tuple(t.clone() for t in s["initial"])
        s["sim"] = L.MultimaterialSimulator(layout=_layout(case))
        for m in range(2):
            s["sim"].add_material(s["grids"][m], s["grids"][2 + m],
                                  _options(case, gamma=gammas[m]))
    elif case["kind"] == "batch":
        from fluidity_amd import batch as B
        grids = _batch_input(case, seed)
        s["grids"] = [U for U, _ in grids]
        s["batch"] = B.Batch([{"U": U, "scheme": _options(case, gamma=g), "cfl": CFL,
                               "dh": 1.0 / n[-1]}
                              for (U, g), n in zip(grids, _batch_sizes(case))],
                             layout=_layout(case))
    else:
        from fluidity_amd import adjoint as A
        s["U"], s["target"] = _adjoint_input(case, seed)
        s["adjoint"] = A.Adjoint(_options(case, gamma=GAMMA, bc="periodic"), CFL,
                                 1.0 / case["nx"], layout=_layout(case))
    return s


def run(s):
    case = s["case"]
    if case["kind"] == "gas":
        r = s["solver"].simulate(s["U"], s["work"], CFL, 1.0 / case["nx"],
                                 max_iters=case["steps"])
        return {"U": s["U"], "run_time": r.run_time, "iters": r.iters,
                "max_wavespeed": r.max_wavespeed}
    if case["kind"] == "bubble":
        for grid, initial in zip(s["grids"], s["initial"]):
            grid.copy_(initial)
        r = s["sim"].simulate_mm(CFL, 1.0 / case["ny"], max_iters=case["steps"],
                                 reinit_every=case["reinit"])
        return {"grids": list(s["grids"]), "run_time": r.run_time, "iters": r.iters}
    if case["kind"] == "batch":
        s["batch"].step(case["steps"])
        results = s["batch"].finish()
        return {"grids": list(s["grids"]), "run_time": torch.tensor([r.run_time for r in results],
                                                                    dtype=torch.float64)}
    U = s["U"].clone()
    done = s["adjoint"].forward(U, case["steps"], checkpoint_every=case["every"])
    grad = torch.zeros_like(U)
    rho = U[..., 0] if case["layout"] == "aos" else U[0]
    (grad[..., 0] if case["layout"] == "aos" else grad[0]).copy_(rho - s["target"])
    dgamma = s["adjoint"].backward(grad, done)
    return {"U": U, "grad": grad, "dgamma": dgamma}


def work(case):
    """A step's time step comes from the maximum over the whole grid, so each
    step reads and writes the state once.  Operations: those of the scheme's
    formulas, about 280 per cell and sweep."""
    def gas(cells, nd, steps, size):
        return steps * cells * 2 * (2 + nd) * size, steps * cells * nd * 280.0

    if case["kind"] == "gas":
        nd = 2 if case["ny"] else 1
        b, f = gas(case["nx"] * (case["ny"] or 1), nd, case["steps"],
                   4 if case["dtype"] == "f32" else 8)
    elif case["kind"] == "bubble":
        cells = case["nx"] * case["ny"]
        b, f = gas(2 * cells, 2, case["steps"], 8)
        # both level sets read and written, and three stages of about 150
        # operations per level set
        b += case["steps"] * cells * 2 * 16
        f += case["steps"] * cells * 2 * 3 * 150.0
    elif case["kind"] == "batch":
        b = f = 0
        for shape in _batch_sizes(case):
            x = gas(math.prod(shape), len(shape), case["steps"], 4 if case["dtype"] == "f32" else 8)
            b, f = b + x[0], f + x[1]
    else:
        # forward, and back: the states once more and the adjoint read and
        # written; the reverse of a step costs about three times the step
        cells = case["nx"] * case["ny"]
        b, f = gas(cells, 2, case["steps"], 8)
        b, f = b + case["steps"] * cells * 3 * 32, f * 4
    return {"bytes": float(b), "flops": float(f)}


# ---------------------------------------------------------------------------
# the same results in 64 bits, in plain torch
# ---------------------------------------------------------------------------

def _pad(U, bc):
    """U (S, ..) with PAD ghost cells on every side of every dimension."""
    nd = U.dim() - 1
    for d in range(nd):
        axis = U.dim() - 1 - d
        n = U.shape[axis]
        i = torch.arange(-PAD, n + PAD, device=U.device)
        ghost = (i < 0) | (i >= n)
        if bc == "periodic":
            i = i % n
        else:
            i = torch.where(i < 0, -i - 1, torch.where(i >= n, 2 * n - 1 - i, i))
        U = U.index_select(axis, i)
        if bc == "reflective":
            sign = torch.where(ghost, -1.0, 1.0).double()
            sign = sign.view([-1 if a == axis - 1 else 1 for a in range(nd)])
            U = torch.stack([U[k] * sign if k == 2 + d else U[k] for k in range(U.shape[0])])
    return U


def _at(t, k, d):
    """t at offset k along dimension d (x is 0); wraps, in the ghost cells only."""
    return torch.roll(t, -k, t.dim() - 1 - d)


def _prim(U, gamma):
    v = [U[2 + i] / U[0] for i in range(U.shape[0] - 2)]
    return v, (gamma - 1.0) * (U[1] - 0.5 * U[0] * sum(a * a for a in v))


def _flux(U, v, p, D):
    F = [m * v[D] for m in U]
    F[0] = U[2 + D]
    F[1] = v[D] * (U[1] + p)
    F[2 + D] = U[2 + D] * v[D] + p
    return F


def _flattening(v, p):
    """The slopes' factor: 1, or less at strong shocks, from both dimensions."""
    chi = torch.ones_like(p)
    for d in range(len(v)):
        jump = _at(p, 1, d) - _at(p, -1, d)
        dp = jump.abs()
        wide = (_at(p, 2, d) - _at(p, -2, d)).abs()
        shock = (_at(v[d], -1, d) > _at(v[d], 1, d)) & \
            (dp / torch.minimum(_at(p, 1, d), _at(p, -1, d)) > 0.33)
        z = dp / torch.where(wide > 0, wide, torch.ones_like(wide))
        K = torch.where(wide > 0, 1.0 - (z - 0.75) / (0.85 - 0.75), torch.zeros_like(z))
        K = torch.where(shock, K.clamp(0.0, 1.0), torch.ones_like(K))
        beside = torch.where(jump > 0, _at(K, 1, d), torch.where(jump < 0, _at(K, -1, d), K))
        chi = torch.minimum(chi, torch.minimum(K, beside))
    return chi


def _limit(b, f, limiter):
    """The limiter of the ratio b / f."""
    ok = f != 0
    r = torch.where(ok, b / torch.where(ok, f, torch.ones_like(f)), torch.zeros_like(f))
    pos = r > 0
    r = torch.where(pos, r, torch.ones_like(r))
    if limiter == "superbee":
        v = torch.where(r <= 0.5, 2.0 * r,
                        torch.where(r <= 1.0, torch.ones_like(r),
                                    torch.minimum(2.0 / (1.0 + r), r.clamp(max=2.0))))
    else:
        v = 2.0 * r.clamp(max=1.0) / (1.0 + r)
    return torch.where(pos, v, torch.zeros_like(v))


def _hllc(ul, ur, gamma, D):
    (vl, pl), (vr, pr) = _prim(ul, gamma), _prim(ur, gamma)
    al, ar = torch.sqrt(gamma * pl / ul[0]), torch.sqrt(gamma * pr / ur[0])
    ps = 0.5 * (pl + pr - 0.25 * (vr[D] - vl[D]) * (ur[0] + ul[0]) * (al + ar))
    ps = ps.clamp(min=0.0)
    q = (gamma + 1.0) / (2.0 * gamma)

    def speed(u, p, a):
        shock = ps > p
        return u + a * torch.sqrt(1.0 + q * torch.where(shock, ps / p - 1.0, torch.zeros_like(p)))
    sl, sr = speed(vl[D], pl, -al), speed(vr[D], pr, ar)
    kl, kr = ul[0] * (sl - vl[D]), ur[0] * (sr - vr[D])
    star = (pr - pl + vl[D] * kl - vr[D] * kr) / (kl - kr)
    Fl, Fr = _flux(ul, vl, pl, D), _flux(ur, vr, pr, D)

    def beyond(u, v, p, s, F):
        c = (s - v[D]) / (s - star)
        us = [m * c for m in u]
        us[2 + D] = star * u[0] * c
        us[1] = c * (u[1] + u[0] * (star - v[D]) * (star + p / (u[0] * (s - v[D]))))
        return [F[k] + (us[k] - u[k]) * s for k in range(len(F))]
    Sl, Sr = beyond(ul, vl, pl, sl, Fl), beyond(ur, vr, pr, sr, Fr)
    return [torch.where(sl >= 0, Fl[k], torch.where(sr <= 0, Fr[k],
                                                    torch.where(star >= 0, Sl[k], Sr[k])))
            for k in range(len(Fl))]


def _force(ul, ur, gamma, D, dtdh):
    Fl, Fr = _flux(ul, *_prim(ul, gamma), D), _flux(ur, *_prim(ur, gamma), D)
    S = range(len(Fl))
    mid = torch.stack([0.5 * (ul[k] + ur[k] + (Fl[k] - Fr[k]) * dtdh) for k in S])
    Fm = _flux(mid, *_prim(mid, gamma), D)
    return [0.5 * (0.5 * (Fl[k] + Fr[k] + (ul[k] - ur[k]) / dtdh) + Fm[k]) for k in S]


def _sweep(U, gamma, dtdh, D, case, bc):
    P = _pad(U, bc)
    v, p = _prim(P, gamma)
    chi = _flattening(v, p)
    back, ahead = P - _at(P, -1, D), _at(P, 1, D) - P
    if case.get("form") == "prim":
        W = torch.stack([P[0], p] + v)
        b, f = W - _at(W, -1, D), _at(W, 1, D) - W
    else:
        b, f = back, ahead
    delta = 0.25 * chi * (back + ahead) * _limit(b, f, case.get("limiter"))
    plus, minus = P + delta, P - delta
    half = 0.5 * dtdh * (torch.stack(_flux(minus, *_prim(minus, gamma), D)) -
                         torch.stack(_flux(plus, *_prim(plus, gamma), D)))
    R, L = plus + half, _at(minus + half, 1, D)
    G = torch.stack(_force(R, L, gamma, D, dtdh) if case.get("flux") == "force"
                    else _hllc(R, L, gamma, D))
    out = P + dtdh * (_at(G, -1, D) - G)
    for d in range(U.dim() - 1):
        axis = U.dim() - 1 - d
        out = out.narrow(axis, PAD, U.shape[axis])
    return out


def _speed(U, gamma):
    v, p = _prim(U, gamma)
    most = v[0].abs()
    for a in v[1:]:
        most = torch.maximum(most, a.abs())
    return (most + torch.sqrt(gamma * p / U[0])).max()


def _step(U, gamma, dh, case, bc, dt=None):
    """(new state, dt)"""
    dt = CFL * dh / _speed(U, gamma) if dt is None else dt
    for D in range(U.dim() - 1):
        U = _sweep(U, gamma, dt / dh, D, case, bc)
    return U, dt


def _loop(U, gamma, dh, case, bc):
    t = 0.0
    for _ in range(case["steps"]):
        U, dt = _step(U, gamma, dh, case, bc)
        t = t + dt
    return U, float(t)


def _gather(A, y, x):
    """A (.., ny, nx) at mirrored cell indices y, x."""
    def mirror(i, n):
        i = torch.where(i < 0, -i - 1, i)
        return torch.where(i >= n, 2 * n - 1 - i, i).clamp(0, n - 1)
    return A[..., mirror(y, A.shape[-2]), mirror(x, A.shape[-1])]


def _beside(phi, d, k):
    """phi one cell along d; the edge cell repeats."""
    axis = 1 - d
    i = (torch.arange(phi.shape[axis], device=phi.device) + k).clamp(0, phi.shape[axis] - 1)
    return phi.index_select(axis, i)


def _normal(phi, dh):
    g = [(_beside(phi, d, 1) - _beside(phi, d, -1)) * (0.5 / dh) for d in range(2)]
    mag = torch.sqrt(g[0] * g[0] + g[1] * g[1])
    return [torch.where(mag == 0, torch.zeros_like(a), a / torch.where(mag == 0, 1.0, mag))
            for a in g]


def _star(phi, other, U, V, gu, gv, dh):
    """U with the star states of the Riemann problem across the interface at
    the cells just inside it."""
    take = (phi <= 0) & (phi >= -dh) & (other >= 0) & (other < dh)
    for d in range(2):
        take = take & (_beside(phi, d, 1) != 0) & (_beside(phi, d, -1) != 0)
    y, x = torch.nonzero(take, as_tuple=True)
    n = [a[y, x] for a in _normal(phi, dh)]
    depth = phi[y, x].abs()

    def probe(A, dist):
        o, f = [], []
        for d in range(2):
            w = n[d] * dist / dh
            whole = torch.floor(w.abs())
            o.append([(torch.sign(w) * whole).long(),
                      (torch.sign(w) * whole).long() + torch.sign(w).long()])
            f.append(w.abs() - whole)
        a, b = _gather(A, y + o[1][0], x + o[0][0]), _gather(A, y + o[1][0], x + o[0][1])
        c, e = _gather(A, y + o[1][1], x + o[0][0]), _gather(A, y + o[1][1], x + o[0][1])
        near, far = a * (1 - f[0]) + b * f[0], c * (1 - f[0]) + e * f[0]
        return near * (1 - f[1]) + far * f[1]
    wl, wr = probe(U, depth - 1.5 * dh), probe(V, depth + 1.5 * dh)
    (vl, pl), (vr, pr) = _prim(wl, gu), _prim(wr, gv)
    rl, rr = wl[0], wr[0]
    nl, nr = vl[0] * n[0] + vl[1] * n[1], vr[0] * n[0] + vr[1] * n[1]
    al, ar = torch.sqrt(gu * pl / rl), torch.sqrt(gv * pr / rr)
    ps = (0.5 * (pl + pr - 0.25 * (nr - nl) * (rr + rl) * (al + ar))).clamp(min=0.0)

    def speed(u, p, a, g):
        return u + a * torch.sqrt(1.0 + (g + 1.0) / (2.0 * g) * (ps / p - 1.0).clamp(min=0.0))
    sl, sr = speed(nl, pl, -al, gu), speed(nr, pr, ar, gv)
    kl, kr = rl * (sl - nl), rr * (sr - nr)
    s = (pr - pl + nl * kl - nr * kr) / (kl - kr)
    c = (sl - nl) / (sl - s)
    E = pl / (gu - 1.0) + 0.5 * rl * nl * nl
    rho, E = rl * c, c * (E + rl * (s - nl) * (s + pl / (rl * (sl - nl))))
    p = (gu - 1.0) * (E - 0.5 * rho * s * s)
    out = U.clone()
    out[:, y, x] = _cons(torch.stack([rho, p] + [vl[d] + (s - nl) * n[d] for d in range(2)]), gu)
    return out


def _extrapolate(phi, U, A, dh, sweeps=8):
    """U with its ghost band filled from the field A, which holds star states."""
    band = (phi > 0) & (phi <= 6.0 * dh / math.sqrt(2.0))
    n = [a.abs() for a in _normal(phi, dh)]
    l1 = n[0] + n[1]
    steep = l1 > 1e-2
    down = [_beside(phi, d, -1) < _beside(phi, d, 1) for d in range(2)]
    for _ in range(sweeps):
        acc = 0.0
        for d in range(2):
            up = torch.stack([torch.where(down[d], _beside(a, d, -1), _beside(a, d, 1)) for a in A])
            acc = acc + up * torch.where(steep, n[d], torch.full_like(l1, 0.5))
        A = torch.where(band, acc / torch.where(steep, l1, torch.ones_like(l1)), A)
    return torch.where(band, A, U)


def _weno(d1, d2, d3, d4, d5):
    e = 1e-5 * torch.stack([d1 * d1, d2 * d2, d3 * d3, d4 * d4, d5 * d5]).amax(0) + 1e-98
    a = [w / (13.0 / 12.0 * s * s + 0.25 * t * t + e) ** 2 for w, s, t in (
        (0.1, d1 - 2 * d2 + d3, d1 - 4 * d2 + 3 * d3), (0.6, d2 - 2 * d3 + d4, d2 - d4),
        (0.3, d3 - 2 * d4 + d5, 3 * d3 - 4 * d4 + d5))]
    return (a[0] * (2 * d1 - 7 * d2 + 11 * d3) + a[1] * (-d2 + 5 * d3 + 2 * d4) +
            a[2] * (2 * d3 + 5 * d4 - d5)) / (6.0 * (a[0] + a[1] + a[2]))


def _rate(phi, V, dh):
    """V |grad phi|, fifth order and upwind."""
    total = 0.0
    for d in range(2):
        axis, n = 1 - d, phi.shape[1 - d]
        i = torch.arange(-3, n + 3, device=phi.device)
        i = torch.where(i < 0, -i - 1, torch.where(i >= n, 2 * n - 1 - i, i))
        f = phi.index_select(axis, i)
        f = [f.narrow(axis, k, n) for k in range(7)]
        g = [(f[k + 1] - f[k]) / dh for k in range(6)]
        b, a = _weno(*g[:5]), _weno(*g[:0:-1])
        left = V <= 0
        b = torch.where(left, b.clamp(min=0.0), b.clamp(max=0.0))
        a = torch.where(left, a.clamp(max=0.0), a.clamp(min=0.0))
        total = total + torch.maximum(a * a, b * b)
    return V * torch.sqrt(total)


def _redistance(phi, dh, band=6):
    """Signed distance within `band` cells of the interface."""
    far = 1e300
    sg = torch.sign(phi)
    source = torch.zeros_like(phi, dtype=torch.bool)
    for d in range(2):
        for k in (-1, 1):
            o = _beside(phi, d, k)
            source = source | ((torch.sign(o) != sg) & (phi.abs() < o.abs()))
    dist = torch.where(source, phi.abs(), torch.full_like(phi, far))
    edge = [[torch.zeros_like(source) for _ in range(2)] for _ in range(2)]
    for d in range(2):
        edge[d][0].select(1 - d, 0).fill_(True)
        edge[d][1].select(1 - d, -1).fill_(True)
    while True:
        best = []
        for d in range(2):
            m = torch.full_like(phi, far)
            for j, k in enumerate((-1, 1)):
                o = _beside(dist, d, k)
                o = torch.where((_beside(sg, d, k) == sg) | (o == far), o, -o)
                m = torch.minimum(m, torch.where(edge[d][j], torch.full_like(o, far), o))
            best.append(m)
        a, b = best
        gap = a - b
        q = torch.where(gap.abs() >= dh, torch.minimum(a, b) + dh,
                        0.5 * (a + b + torch.sqrt((2.0 * dh * dh - gap * gap).clamp(min=0.0))))
        new = torch.where(~source & (q < dist) & (q <= band * dh), q, dist)
        if torch.equal(new, dist):
            break
        dist = new
    return sg * torch.where(dist <= band * dh, dist, torch.full_like(dist, (band + 1) * dh))


def _bubble_exact(case, seed):
    U0, U1, phi, gammas = _bubble_input(case, seed)
    U = [_planes(U0, case["layout"]), _planes(U1, case["layout"])]
    phis, dh, t = [-phi, phi], 1.0 / case["ny"], 0.0
    for k in range(case["steps"]):
        A = [_star(phis[m], phis[1 - m], U[m], U[1 - m], gammas[m], gammas[1 - m], dh)
             for m in range(2)]
        U = [_extrapolate(phis[m], U[m], A[m], dh) for m in range(2)]
        dt = CFL * dh / max(_speed(U[m], gammas[m]) for m in range(2))
        U = [_step(U[m], gammas[m], dh, case, "transmissive", dt)[0] for m in range(2)]
        here = torch.where(phis[0] <= 0, U[0], U[1])
        u = [here[2 + d] / here[0] for d in range(2)]
        some = (phis[0] <= 0) | (phis[1] <= 0)
        new = []
        for m in range(2):
            n = _normal(phis[m], dh)
            V = torch.where(some, u[0] * n[0] + u[1] * n[1], torch.zeros_like(phi))
            f = phis[m]
            a = f - dt * _rate(f, V, dh)
            b = 0.75 * f + 0.25 * (a - dt * _rate(a, V, dh))
            new.append(f / 3.0 + (b - dt * _rate(b, V, dh)) * 2.0 / 3.0)
        half = 0.5 * (new[0] - new[1])
        phis = [half, -half]
        if k % case["reinit"] == case["reinit"] - 1:
            phis = [_redistance(f, dh) for f in phis]
        t = t + dt
    return {"grids": [_laid(A, case["layout"]) for A in U] + phis, "run_time": float(t),
            "iters": None}


def _adjoint_exact(case, seed):
    from torch.utils.checkpoint import checkpoint
    U0, target = _adjoint_input(case, seed)
    U0 = _planes(U0, case["layout"]).clone().requires_grad_(True)
    gamma = torch.tensor(GAMMA, dtype=torch.float64, device="cuda", requires_grad=True)
    U = U0
    for _ in range(case["steps"]):
        U = checkpoint(lambda A, g: _step(A, g, 1.0 / case["nx"], case, "periodic")[0], U, gamma,
                       use_reentrant=False)
    (0.5 * (U[0] - target) ** 2).sum().backward()
    return {"U": _laid(U.detach(), case["layout"]), "grad": _laid(U0.grad, case["layout"]),
            "dgamma": float(gamma.grad)}


def exact(case, seed):
    if case["kind"] == "bubble":
        return _bubble_exact(case, seed)
    if case["kind"] == "adjoint":
        return _adjoint_exact(case, seed)
    if case["kind"] == "batch":
        done = [_loop(_planes(U, case["layout"]), g, 1.0 / n[-1], case, "transmissive")
                for (U, g), n in zip(_batch_input(case, seed), _batch_sizes(case))]
        return {"grids": [_laid(U, case["layout"]) for U, _ in done],
                "run_time": torch.tensor([t for _, t in done], dtype=torch.float64)}
    U, t = _loop(_planes(_gas_input(case, seed), case["layout"]), GAMMA, 1.0 / case["nx"], case,
                 case["bc"])
    return {"U": _laid(U, case["layout"]), "run_time": t, "iters": None,
            "max_wavespeed": float(_speed(U, GAMMA))}
