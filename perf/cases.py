"""The work that a user of this framework has it do, as timed cases.

A program holds a Context (one instance or a batch) or its own device state,
and asks for steps: one at a time, hundreds between two exported frames, a
frame of an app with its moving window and data collection, or a gradient.
Each case is one such request through the public entry points of
fivonagi_amd, with what the program reads back after it.

Sizes are those of the repository's workloads, tests and benchmark
(fivonagi_amd/workloads.py, bench.py) and odd ones between them.  Every state
is a field of wave packets over a weak background, made from the seed.

Interface: listed(), draw(rng), prepare(case, seed), run(state), work(case),
exact(case, seed) (the same outputs from plain torch in 64 bits).
"""
import math

import numpy as np
import torch

import fivonagi_amd as fa
from fivonagi_amd import workloads as wl

DEV = "cuda" if torch.cuda.is_available() else "cpu"

# One step moves a state in and a state out: 3 fields each way.  FP operations
# per cell and step: the two Riemann solves (about 40 each), limiters and
# fluxes (60 each), updates, velocities and source (40).
FLOPS_PER_CELL = 240.0
# reading q_n and the adjoint in, writing the adjoint out; the transposed
# step repeats the forward's arithmetic and about twice more
ADJ_FLOPS_PER_CELL = 700.0


def listed():
    return [
        # a program coupled to the solver step by step: the smallest call,
        # launches and host round trips
        dict(name="step1_128x96", kind="steps", app="edge", nx=128, ny=96, steps=1, fp64=False,
             cfl_all=False, n=1),
        # the 400x400 pulse workload between two frames: an ordinary small
        # grid, whose CFL subset is irregular
        dict(name="pulse_400", kind="steps", app="pulse", nx=400, ny=400, steps=250, fp64=False,
             cfl_all=False, n=1),
        # a serving loop that keeps its state in its own device tensors, on a
        # ragged grid with the exact CFL maximum
        dict(name="noalloc_1021x777", kind="noalloc", app="pulse", nx=1021, ny=777, steps=32,
             fp64=False, cfl_all=True, n=1),
        # one frame of the Taylor-shock study in FP32: 12 small and middle
        # instances (4 resolutions x 3 angles) in one batch, moving window,
        # data collection, the cut rows read each frame
        dict(name="taylor_frame_sweep", kind="taylor", etac=8, angles=3, fp64=False, grids=False),
        # the same study in FP64 (PRECISION=2) up to its finest grid, with
        # the whole grids exported
        dict(name="taylor_frame_fp64", kind="taylor", etac=16, angles=1, fp64=True, grids=True),
        # the headline grid, 800 steps between frames
        dict(name="edge_4096x1024", kind="steps", app="edge", nx=4096, ny=1024, steps=800,
             fp64=False, cfl_all=False, n=1),
        # the driven grid in FP64
        dict(name="edge_2048x1024_fp64", kind="steps", app="edge", nx=2048, ny=1024, steps=400,
             fp64=True, cfl_all=False, n=1),
        # a parameter study: 16 uneven instances (256..1024) in one context
        dict(name="batch_16_uneven", kind="steps", app="batch", nx=256, ny=1024, steps=300,
             fp64=False, cfl_all=False, n=16),
        # one frame of the hifu app at ETAC = 2: aperture packet, moving
        # window, microphones and maxima, the field and the grid exported
        dict(name="hifu_frame_1024x2048", kind="hifu", nx=1024, ny=2048, fp64=False),
        # one gradient of the single-instance adjoint workload's grid, every
        # state of the run kept
        dict(name="adjoint_2048x1024", kind="adjoint", nx=2048, ny=1024, n=1, steps=200, every=0),
        # gradients of a batch whose states would not fit: checkpoints, the
        # segments recomputed
        dict(name="adjoint_8x512_ckpt", kind="adjoint", nx=512, ny=512, n=8, steps=64, every=8),
        # the largest single grid, zero-gradient edges
        dict(name="pulse_8192x4096", kind="steps", app="pulse", nx=8192, ny=4096, steps=240,
             fp64=False, cfl_all=False, n=1),
    ]


def _size(rng, lo, hi):
    """Log-uniform, odd as often as even."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["steps", "steps", "steps", "noalloc", "taylor", "hifu", "adjoint"])
    if kind == "taylor":
        return dict(kind=kind, etac=rng.choice([3, 5, 6, 7, 9, 10, 11, 12, 13]),
                    angles=rng.choice([1, 2, 3, 4]), fp64=rng.random() < 0.5,
                    grids=rng.random() < 0.5)
    if kind == "hifu":
        nx = _size(rng, 96, 2048)
        return dict(kind=kind, nx=nx, ny=min(2 * nx + rng.randrange(-9, 10), 4096),
                    fp64=rng.random() < 0.4)
    if kind == "adjoint":
        nx, ny = _size(rng, 64, 2048), _size(rng, 64, 1536)
        return dict(kind=kind, nx=nx, ny=ny, n=rng.choice([1, 1, 2, 4]),
                    steps=rng.randrange(12, 160), every=rng.choice([0, 0, 1, 5, 12]))
    nx, ny = _size(rng, 40, 4500), _size(rng, 40, 3000)
    steps = max(1, min(_size(rng, 1, 700), int(4e9 / (nx * ny))))
    if kind == "noalloc":
        return dict(kind=kind, app=rng.choice(["edge", "pulse"]), nx=nx, ny=ny,
                    steps=min(steps, 128), fp64=False, cfl_all=rng.random() < 0.5, n=1)
    app = rng.choice(["edge", "pulse", "batch"])
    n = 1
    if app == "batch":
        n = rng.randrange(2, 20)
        nx, ny = sorted((_size(rng, 64, 1100), _size(rng, 64, 1100)))
        steps = min(steps, 300)
    return dict(kind=kind, app=app, nx=nx, ny=ny, steps=steps, fp64=rng.random() < 0.35,
                cfl_all=rng.random() < 0.3, n=n)


# ------------------------------------------------------------------ inputs --

def _field(rng, nx, ny, amp=8e-3, scale=1.0):
    """(3, ny, nx) float64: linear wave packets (rho', rho u, rho v) of random
    place, direction, wavelength and width over a weak background wave.  scale:
    lengths in units of the default 20 cells per wavelength."""
    x = torch.arange(nx, dtype=torch.float64, device=DEV)[None, :]
    y = torch.arange(ny, dtype=torch.float64, device=DEV)[:, None]
    q = torch.zeros((3, ny, nx), dtype=torch.float64, device=DEV)

    def add(r, th, ys, xs):
        q[0, ys, xs] += r
        q[1, ys, xs] += r * math.cos(th)
        q[2, ys, xs] += r * math.sin(th)

    every = slice(None)
    for _ in range(3):
        th, k = rng.uniform(0, 2 * math.pi), 2 * math.pi / (scale * rng.uniform(40, 90))
        ph = rng.uniform(0, 2 * math.pi)
        add(0.02 * amp * torch.sin(k * (x * math.cos(th) + y * math.sin(th)) + ph), th, every,
            every)
    for _ in range(int(min(64, max(3, nx * ny / 2e4)))):
        th, k = rng.uniform(0, 2 * math.pi), 2 * math.pi / (scale * rng.uniform(18, 36))
        w = scale * rng.uniform(15, 60)
        cx, cy = rng.uniform(0, nx), rng.uniform(0, ny)
        a = amp * rng.uniform(0.15, 1.0)
        xs = slice(max(0, int(cx - 4 * w)), min(nx, int(cx + 4 * w) + 1))
        ys = slice(max(0, int(cy - 4 * w)), min(ny, int(cy + 4 * w) + 1))
        if xs.start >= xs.stop or ys.start >= ys.stop:
            continue
        dx, dy = x[:, xs] - cx, y[ys] - cy
        add(a * torch.sin(k * (dx * math.cos(th) + dy * math.sin(th)))
            * torch.exp(-(dx * dx + dy * dy) / (2 * w * w)), th, ys, xs)
    return q.cpu().numpy()


def _taylor_at(p, T):
    """The Taylor instance p at time T: the front in the grid, the window about
    to move (it starts at T = 6.25 / cos(theta))."""
    t = p.taylor
    x = np.arange(p.nx)[None, :] * p.dx
    y = (np.arange(p.ny)[:, None] - t["jc"]) * p.dy + t["yoff"]
    cs, sn = math.cos(t["theta"]), math.sin(t["theta"])
    r = t["rhoa"] * np.tanh(t["c"] * (x * cs + y * sn - T))
    return fa.Problem(p.nx, p.ny, p.dx, p.dy, p.beta, p.delta, np.stack([r, r * cs, r * sn]),
                      cfl_wish=p.cfl_wish, dt0=p.dt0, T0=T, bc=p.bc, taylor=t, moving=p.moving)


def _problems(case, seed):
    """The case's fa.Problem objects, from the seed alone."""
    rng = np.random.default_rng(seed)
    d = 1.0 / wl.CELLS_PER_UNIT
    kind = case["kind"]
    mode = fa.CFL_ALL if case.get("cfl_all") else fa.CFL_REFERENCE_FOLD

    def edge(nx, ny, delta):
        hw = ny * rng.uniform(0.15, 0.3)
        amp = wl.edge_profile(ny, 0.02, hw) + 4e-4 * (1 + 0.3 * rng.standard_normal(ny))
        phase = 0.05 * rng.standard_normal(ny)
        omega = 2 * math.pi * wl.CELLS_PER_UNIT / rng.uniform(18.0, 30.0)
        return fa.Problem(nx, ny, d, d, rng.uniform(3.0, 4.0), delta, _field(rng, nx, ny, 2e-3),
                          bc=fa.BC_EDGE_DRIVE, cfl_mode=mode, omega=omega, edge_amp=amp,
                          edge_phase=phase)

    def pulse(nx, ny):
        return fa.Problem(nx, ny, d, d, rng.uniform(3.0, 4.0), 10 ** rng.uniform(-4.5, -3.5),
                          _field(rng, nx, ny), bc=fa.BC_ZEROGRAD, cfl_mode=mode)

    if kind == "taylor":
        # the study's instances: resolutions up to etac by halving, angles of
        # its sweep, the amplitude (delta / beta) from the seed
        etas = sorted({max(1, case["etac"] >> k) for k in range(4)})
        angles = [0.0, math.pi / 16, math.pi / 4, math.pi / 8][:case["angles"]]
        return [_taylor_at(wl.taylor(e, theta=th, delta=1e-7 * rng.uniform(0.5, 2.0),
                                     moving=True, cflw=float(rng.choice([0.6, 0.7, 0.8, 0.9]))),
                           5.0)
                for e in etas for th in angles]
    if kind == "hifu":
        p = wl.hifu(nx=case["nx"], ny=case["ny"], ispam=float(rng.choice([10.0, 20.0, 30.0])))
        # the frames after the packet's start: waves already in the window
        q = _field(rng, p.nx, p.ny, amp=4e-4, scale=p.nx / 25.0 / 20.0)
        p = fa.Problem(p.nx, p.ny, p.dx, p.dy, p.beta, p.delta, q, dt0=p.dt0, T0=1.0, bc=p.bc,
                       moving=p.moving, hifu=p.hifu)
        return [p]
    if kind == "adjoint":
        return [edge(case["nx"], case["ny"], 1e-4) for _ in range(case["n"])]
    if case["app"] == "batch":
        # sizes from lo to hi, each paired with its mirror: the same for every seed
        s = np.linspace(case["nx"], case["ny"], case["n"]).astype(int)
        order = np.random.default_rng(case["n"]).permutation(case["n"])
        return [pulse(int(s[k]), int(s[-1 - k])) for k in order]
    return [edge(case["nx"], case["ny"], 5e-5) if case["app"] == "edge"
            else pulse(case["nx"], case["ny"]) for _ in range(case["n"])]


def _box(case):
    """The objective's box: a focus a few wavelengths into the grid."""
    nx, ny = case["nx"], case["ny"]
    w, h = min(64, nx // 3), min(64, ny // 3)
    return (min(24, nx // 3), ny // 2 - h // 2, w, h)


def prepare(case, seed):
    probs = _problems(case, seed)
    kind = case["kind"]
    if kind == "noalloc":
        p = probs[0]
        q = torch.zeros((6, p.ny, p.nx), dtype=torch.float32, device=DEV)
        q[:3] = torch.from_numpy(p.q0).to(DEV)
        return dict(case=case, prob=p, q=q, ptrs=[q[k].data_ptr() for k in range(6)], state=None)
    ctx = fa.Context(probs, fp64=case.get("fp64", False))
    if kind == "taylor":
        for k, p in enumerate(probs):
            ctx.set_collect(k, **wl.taylor_collect(p, ctx.fp64))
    elif kind == "hifu":
        ctx.set_collect(0, **wl.hifu_collect(probs[0]))
    return dict(case=case, ctx=ctx, probs=probs, T=min(p.T0 for p in probs))


def run(state):
    case, kind = state["case"], state["case"]["kind"]
    if kind == "noalloc":
        st = fa.step_noalloc(state["prob"], state["ptrs"], case["steps"], state=state["state"],
                             stream=torch.cuda.current_stream().cuda_stream)
        state["state"] = st
        return dict(q=[state["q"][:3]], n=[st.n_accepted], T=[np.float32(st.T)])
    ctx, probs = state["ctx"], state["probs"]
    if kind == "steps":
        ctx.step(case["steps"])
        got = [ctx.collect(k) for k in range(len(probs))]
        return dict(q=[g[0] for g in got], n=[g[1]["n_accepted"] for g in got],
                    T=[np.float32(g[1]["T"]) for g in got])
    if kind in ("taylor", "hifu"):
        state["T"] += 1.0                       # DTPRINT
        ctx.step_until(state["T"])
        info = [ctx.info(k) for k in range(len(probs))]
        out = dict(n=[i["n_accepted"] for i in info],
                   measure=[ctx.measure(k, rows=4 if kind == "taylor" else None)
                            for k in range(len(probs))])
        if kind == "hifu" or case["grids"]:
            out["q"] = [ctx.collect(k)[0] for k in range(len(probs))]
        return out
    # the adjoint runs in FP32: J and the gradients as an optimiser in that
    # precision holds them
    J, ga, gp = ctx.step_adjoint(case["steps"], [_box(case)] * len(probs),
                                 checkpoint_every=case["every"])
    got = [ctx.collect(k) for k in range(len(probs))]
    return dict(J=J.astype(np.float32), ga=[g.astype(np.float32) for g in ga],
                gp=[g.astype(np.float32) for g in gp], q=[g[0] for g in got],
                n=[g[1]["n_accepted"] for g in got])


def work(case):
    kind = case["kind"]
    size = 8 if case.get("fp64") else 4
    if kind == "taylor":
        b = f = 0.0
        for e in sorted({max(1, case["etac"] >> k) for k in range(4)}):
            cells, steps = (64.0 * e) ** 2, 1.0 / (0.75 * 12.5 / (64 * e - 1))
            b += case["angles"] * cells * steps * 6 * size
            f += case["angles"] * cells * steps * FLOPS_PER_CELL
        return dict(bytes=b, flops=f)
    if kind == "hifu":
        cells = float(case["nx"]) * case["ny"]
        steps = 1.0 / (0.9 * 25.0 / (case["nx"] - 1))
        return dict(bytes=cells * steps * 6 * size, flops=cells * steps * FLOPS_PER_CELL)
    if kind == "adjoint":
        cells = float(case["nx"]) * case["ny"] * case["n"] * case["steps"]
        return dict(bytes=cells * (24 + 36), flops=cells * (FLOPS_PER_CELL + ADJ_FLOPS_PER_CELL))
    if case["app"] == "batch":
        s = np.linspace(case["nx"], case["ny"], case["n"]).astype(int)
        cells = float((s * s[::-1]).sum())
    else:
        cells = float(case["nx"]) * case["ny"] * case["n"]
    return dict(bytes=cells * case["steps"] * 6 * size,
                flops=cells * case["steps"] * FLOPS_PER_CELL)


# ---------------------------------------------- the same in 64 bits, torch --

def _fold_cells(nx, ny):
    """Flat indexes whose value the reference's reduction carries to cfl[0]."""
    N = nx * ny
    strides, s = [], N
    while s > 32:
        s //= 2
        strides.append((s // 16) * 16)
    while s > 2:
        s //= 2
        strides.append(s)
    m = torch.zeros(N, dtype=torch.bool, device=DEV)
    m[0] = True
    for S in reversed(strides):
        k = min(S, N - S)
        if k > 0:
            m[S:S + k] |= m[:k].clone()
    return m


class _Exact:
    """The step in 64 bits: boundary, y sweep, x sweep, source, dt rule."""

    def __init__(self, p, fp64):
        self.p = p
        self.q = torch.from_numpy(p.q0_f64 if fp64 else p.q0).to(DEV).double()
        self.T, self.dt = p.T0, p.dt0
        self.n = self.mdx = self.mdy = 0
        self.mask = None if p.cfl_mode == fa.CFL_ALL else _fold_cells(p.nx, p.ny)
        self.log = []

    def boundary(self, q, T, amp=None, phase=None):
        p, nx, ny = self.p, self.p.nx, self.p.ny
        b = q.clone()
        if p.bc == fa.BC_TAYLOR:
            t = p.taylor
            i = torch.arange(nx, dtype=torch.float64, device=DEV)[None, :] + self.mdx
            j = torch.arange(ny, dtype=torch.float64, device=DEV)[:, None] + self.mdy
            cs, sn = math.cos(t["theta"]), math.sin(t["theta"])
            r = t["rhoa"] * torch.tanh(t["c"] * (i * p.dx * cs
                                                 + ((j - t["jc"]) * p.dy + t["yoff"]) * sn - T))
            g = torch.stack([r, r * cs, r * sn])
            g[:, 2:-2, 2:-2] = q[:, 2:-2, 2:-2]
            return g
        b[:, :, nx - 2:] = q[:, :, nx - 3:nx - 2]
        if p.bc == fa.BC_HIFU:
            h = p.hifu
            b[:, ny - 2:, :] = q[:, ny - 3:ny - 2, :]
            b[:, :, :2] = q[:, :, 2:3]
            width = min(int(h["a"] / p.dy), ny - 2)
            if self.mdx == 0 and width > 0:
                jp = torch.arange(width, dtype=torch.float64, device=DEV)
                nd = torch.sqrt(jp * jp + h["f"] ** 2)
                phi = p.dx * jp * jp / (2 * h["f"])
                pack = (h["ampl"] * torch.sin(2 * math.pi * h["frec"] * (T + phi))
                        * torch.exp(-(h["frec"] * (T + phi) / 4) ** 10))
                v = torch.stack([pack, h["f"] / nd * pack * (pack + 1), -jp / nd * pack * (pack + 1)])
                b[:, 2:2 + width, :2] = v[:, :, None]
            b[:, 0, :], b[:, 1, :] = q[:, 4, :], q[:, 3, :]
            b[2, :2, :] = -b[2, :2, :]
            for ys in (slice(0, 2), slice(ny - 2, ny)):
                for xs in (slice(0, 2), slice(nx - 2, nx)):
                    b[:, ys, xs] = 0
            return b
        b[:, :2, :] = q[:, 2:3, :]
        b[:, ny - 2:, :] = q[:, ny - 3:ny - 2, :]
        b[:, :, :2] = q[:, :, 2:3]
        if p.bc == fa.BC_EDGE_DRIVE and self.mdx == 0:
            if amp is None:
                amp = torch.from_numpy(p.edge_amp).to(DEV)
                phase = (torch.zeros_like(amp) if p.edge_phase is None
                         else torch.from_numpy(p.edge_phase).to(DEV))
            d = amp * torch.sin(p.omega * T + phase)
            left = torch.stack([d, d * (d + 1), torch.zeros_like(d)])[:, :, None].expand(3, ny, 2)
            b = torch.cat([left, b[:, :, 2:]], dim=2)
        return b

    def sweep(self, q, axis, dtd, cfl):
        """One directional sweep; cfl: per cell, updated (None: not wanted)."""
        dim = 2 if axis == 0 else 1          # of a (3, ny, nx) tensor
        fn, ft = (1, 2) if axis == 0 else (2, 1)
        N = q.shape[dim]

        def cut(a, lo, n):
            return a.narrow(a.dim() - (1 if axis == 0 else 2), lo, n)

        r1, qn, qt = q[0], q[fn], q[ft]
        un, ut = qn / (1 + r1), qt / (1 + r1)
        L = lambda a: cut(a, 0, N - 1)       # noqa: E731  interface k (1..N-1): cell k-1
        R = lambda a: cut(a, 1, N - 1)       # noqa: E731  and cell k
        Z1m = (L(r1) + R(r1)) / 2
        Z1, Z2, Z3 = Z1m + 1, (L(un) + R(un)) / 2, (L(ut) + R(ut)) / 2
        dr, dn, dtg = R(r1) - L(r1), R(qn) - L(qn), R(qt) - L(qt)
        l3 = Z2 / Z1
        sq = torch.sqrt(l3 * l3 - 2 * Z2 * l3 + 1 + 2 * (self.p.beta - 1) * Z1m)
        l1, l2 = l3 + sq, l3 - sq
        A1 = Z3 * (l1 - 2 * Z2) / (l1 * Z1 - Z3)
        A2 = Z3 * (l2 - 2 * Z2) / (l2 * Z1 - Z3)
        a1 = (dn - dr * l2) / (2 * sq)
        a2 = dr - a1
        a3 = dtg - (a1 * A1 + a2 * A2)
        waves = [(l1, (a1, a1 * l1, a1 * A1)), (l2, (a2, a2 * l2, a2 * A2)), (l3, (a3,))]
        if cfl is not None:
            c = (l3.abs() + sq) * dtd
            if axis == 1:
                cfl[1:] = c
            else:
                cfl[:, 1:] = torch.maximum(cfl[:, 1:], c)
                cfl[:, 0] = 0
        # fluxes of interfaces 2..N-2 (index k - 1 of the arrays above)
        M_ = N - 3
        mid = lambda a: cut(a, 1, M_)        # noqa: E731
        P, M = [0.0, 0.0, 0.0], [0.0, 0.0, 0.0]
        for lam, W in waves:
            s = mid(lam)
            wn = sum(mid(w) * mid(w) for w in W)
            dl = sum(mid(w) * cut(w, 0, M_) for w in W)
            dR = sum(mid(w) * cut(w, 2, M_) for w in W)
            live = wn != 0
            r = torch.where(s > 0, dl, dR) / torch.where(live, wn, torch.ones_like(wn))
            phi = torch.relu(torch.minimum(torch.clamp((1 + r) / 2, max=2.0), 2 * r))
            phi = torch.where(live, phi, torch.zeros_like(phi))   # a zero wave: phi W = 0
            a = s.abs()
            corr = 0.5 * a * (1 - a * dtd) * phi
            pos, neg = torch.relu(s) - corr, -torch.relu(-s) + corr
            for m, w in zip((0, 1, 2) if len(W) == 3 else (2,), W):
                P[m] = P[m] + pos * mid(w)
                M[m] = M[m] + neg * mid(w)
        # cells 2..N-3 of the axis, interior of the other one
        out = q.clone()
        K = N - 4
        inner = (slice(2, -2), slice(None)) if axis == 0 else (slice(None), slice(2, -2))
        for m, f in ((0, 0), (1, fn), (2, ft)):
            flux = cut(P[m], 0, K) + cut(M[m], 1, K)
            cell = cut(q[f], 2, K)
            out[f, 2:-2, 2:-2] = (cell - dtd * flux)[inner]
        return out

    def source(self, q, dt):
        p = self.p
        out = q.clone()
        for f in (1, 2):
            u = q[f] / (1 + q[0])
            c = u[2:-2, 2:-2]
            out[f, 2:-2, 2:-2] = (q[f, 2:-2, 2:-2]
                                  + p.delta * dt / p.dx ** 2 * (u[2:-2, 1:-3] - 2 * c + u[2:-2, 3:-1])
                                  + p.delta * dt / p.dy ** 2 * (u[1:-3, 2:-2] - 2 * c + u[3:-1, 2:-2]))
        return out

    def attempt(self, q, T, dt, cfl, amp=None, phase=None):
        b = self.boundary(q, T, amp, phase)
        b = self.sweep(b, 1, dt / self.p.dy, cfl)
        b = self.sweep(b, 0, dt / self.p.dx, cfl)
        return self.source(b, dt)

    def step(self):
        p = self.p
        while True:
            cfl = torch.zeros_like(self.q[0])
            new = self.attempt(self.q, self.T, self.dt, cfl)
            flat = cfl.reshape(-1)
            c = float((flat if self.mask is None else flat[self.mask]).max())
            dt, ok = self.dt, c < p.cfl_max
            self.dt = dt * p.cfl_wish / c
            if ok:
                break
            self.dt = min(self.dt, 0.9 * dt)
        self.log.append((self.T, dt))
        self.T += dt
        self.n += 1
        if p.moving is not None and self.T >= p.moving[2]:
            vx, vy, t0 = p.moving
            sx = int((self.T - t0) * vx / p.dx) - self.mdx
            sy = int((self.T - t0) * vy / p.dy) - self.mdy
            if sx or sy:
                old = new
                new = old.clone()
                new[:, :p.ny - sy, :p.nx - sx] = old[:, sy:, sx:]
                self.mdx, self.mdy = self.mdx + sx, self.mdy + sy
        self.q = new


def _exact_adjoint(case, p):
    """J and its gradient along the run (dt of each step taken as given)."""
    e = _Exact(p, False)
    states = [e.q]
    for _ in range(case["steps"]):
        e.step()
        states.append(e.q)
    x0, y0, w, h = _box(case)
    amp = torch.from_numpy(p.edge_amp).to(DEV).requires_grad_(True)
    phase = torch.from_numpy(p.edge_phase).to(DEV).requires_grad_(True)
    lam = torch.zeros_like(e.q)
    J = 0.0
    ga, gp = torch.zeros_like(amp), torch.zeros_like(phase)
    for n in reversed(range(case["steps"])):
        T, dt = e.log[n]
        q = states.pop(n).requires_grad_(True)
        new = e.attempt(q, T, dt, None, amp, phase)
        j = dt * new[0, y0:y0 + h, x0:x0 + w].square().sum()
        J += float(j.detach())
        lam, a, b = torch.autograd.grad((new * lam).sum() + j, (q, amp, phase))
        ga += a
        gp += b
    return J, ga.cpu().numpy(), gp.cpu().numpy(), e


def exact(case, seed):
    kind = case["kind"]
    w = work(case)
    if w["flops"] > 3e12 or (kind == "adjoint" and case["steps"] * case["n"] > 600):
        return None                          # longer than is worth waiting for
    probs = _problems(case, seed)
    fp64 = case.get("fp64", False)
    if kind == "adjoint":
        got = [_exact_adjoint(case, p) for p in probs]
        return dict(J=np.array([g[0] for g in got]), ga=[g[1] for g in got],
                    gp=[g[2] for g in got], q=[g[3].q.cpu().numpy() for g in got],
                    n=[g[3].n for g in got])
    es = []
    for p in probs:
        e = _Exact(p, fp64)
        if kind in ("taylor", "hifu"):
            stop = min(x.T0 for x in probs) + 1.0
            while e.T < stop:
                e.step()
        else:
            for _ in range(case["steps"]):
                e.step()
        es.append(e)
    q = [e.q.cpu().numpy() for e in es]
    if kind in ("taylor", "hifu"):
        out = dict(n=[e.n for e in es], measure=[None] * len(es))
        if kind == "hifu" or case["grids"]:
            out["q"] = q
        return out
    return dict(q=q, n=[e.n for e in es], T=[e.T for e in es])
