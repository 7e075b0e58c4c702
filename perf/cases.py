"""Timed workloads of the liquid substep library, as a program that uses it runs them.

Five kinds of work, each through the public entry points:

* "frame": a resident scene advanced by some substeps, then read back for output -- the
  particles (rendering, files) or the grid's face velocities (and in FP64 the pressure).
  Scenes are the repository's dam breaks (block at 8 particles per cell, seeded velocity
  noise) in FP64 or the mixed form, solved with MIC(0)-PCG or AMG-PCG, stepped with
  Scene.substep or with the reference's phase calls, optionally over a resting cloth.
* "exchange": the host owns the particles and hands them over and back each substep, in the
  reference's own arrays (m_x, m_fluid_v, m_fB).
* "rollout": a recorded rollout and its gradients with respect to the initial state.
* "pcg" and "amgpcg": the drop-in pressure solves on a host CSR matrix in the reference's
  bucket-major DOF order.

Downloads go to arrays that the program keeps, as a host program keeps its own.  State of the
mixed form is FP32 on the device, so a program that reads it back stores FP32.
"""
import ctypes

import numpy as np
import torch

import libwetcloth_amd as W
from libwetcloth_amd import scenes

TOL, MAXIT = 1e-6, 2000
PPC = 8


def _frame(name, n, block, **kw):
    """A frame case: n grid cells per axis, block = (y0, x1, y1, z1) of the liquid in units of
    the longest side (x and z start at 0)."""
    c = dict(name=name, kind="frame", nx=n[0], ny=n[1], nz=n[2], y0=block[0], x1=block[1],
             y1=block[2], z1=block[3], sigma=0.5, dt=1.0 / 480, substeps=4, mixed=False,
             amg=False, phases=False, cloth=0, out="grid")
    c.update(kw)
    return c


def listed():
    return [
        # the literal drop-in on the smallest scene the tests run: the host's arrays go over and
        # come back every substep; launches, copies and synchronisations are the cost
        dict(name="exchange_16", kind="exchange", nx=16, ny=16, nz=16, y0=0.0, x1=0.5, y1=0.6,
             z1=1.0, sigma=0.3, dt=1.0 / 480, mixed=False),
        # a small mixed-form simulation rendered from its particles every few substeps
        _frame("frame_32_mixed", (32, 32, 32), (0.0, 0.5, 0.6, 1.0), sigma=0.3, substeps=8,
               mixed=True, out="particles"),
        # the 64^3 FP64 dam break (0.5 M particles), particles read for each output frame
        _frame("frame_64", (64, 64, 64), (0.0, 0.4, 0.6, 1.0), sigma=0.0, substeps=10,
               out="particles"),
        # a long ragged tank: no side a multiple of a bucket or of a tile, stepped by the
        # reference's phase calls
        _frame("ragged_phases", (187, 67, 93), (0.0, 0.61, 0.23, 0.497), dt=1.0 / 960,
               phases=True, substeps=6),
        # the 128^3 dam break (4.0 M particles) in the mixed form
        _frame("frame_128_mixed", (128, 128, 128), (0.0, 0.4, 0.6, 1.0), dt=1.0 / 960, substeps=6,
               mixed=True),
        # the same liquid column resting on a porous cloth: the mixture terms
        _frame("wet_cloth_128", (128, 128, 128), (0.29, 0.4, 0.89, 1.0), dt=1.0 / 960, sigma=0.0,
               substeps=4, mixed=True, cloth=257),
        # the reference's as-shipped solver, FP64
        _frame("frame_128_amg", (128, 128, 128), (0.0, 0.4, 0.6, 1.0), dt=1.0 / 960, substeps=8,
               amg=True),
        # the benchmark: 256^3, 40.3 M particles, in the mixed form and in FP64
        _frame("frame_256_mixed", (256, 256, 256), (0.0, 0.5, 0.6, 1.0), sigma=1.0, dt=1.0 / 1920,
               substeps=4, mixed=True),
        _frame("frame_256", (256, 256, 256), (0.0, 0.5, 0.6, 1.0), sigma=1.0, dt=1.0 / 1920,
               substeps=2),
        # inverse problems: gradients of a short rollout with checkpoints
        dict(name="rollout_32", kind="rollout", nx=32, ny=32, nz=32, y0=0.0, x1=0.5, y1=0.6,
             z1=1.0, sigma=0.3, dt=1.0 / 480, steps=6, every=3),
        # the pressure solve alone from a host program: a block of liquid with an uneven surface
        dict(name="pcg_csr", kind="pcg", nx=51, ny=44, nz=66, tol=1e-8),
        dict(name="amgpcg_csr", kind="amgpcg", nx=64, ny=61, nz=83, tol=1e-8),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["frame"] * 6 + ["exchange", "rollout", "pcg", "amgpcg"])
    if kind in ("pcg", "amgpcg"):
        return dict(kind=kind, nx=_log(rng, 10, 64), ny=_log(rng, 10, 64), nz=_log(rng, 10, 84),
                    tol=rng.choice([1e-6, 1e-8, 1e-10]))
    block = dict(y0=0.0, x1=round(rng.uniform(0.25, 0.6), 3), y1=round(rng.uniform(0.3, 0.7), 3),
                 z1=round(rng.uniform(0.5, 1.0), 3), sigma=round(rng.uniform(0.0, 1.0), 2))
    if kind == "exchange":
        n = _log(rng, 12, 48)
        return dict(kind=kind, nx=n, ny=n, nz=_log(rng, 12, 48), dt=1.0 / 480,
                    mixed=rng.random() < 0.5, **block)
    if kind == "rollout":
        n = _log(rng, 12, 32)
        return dict(kind=kind, nx=n, ny=n, nz=_log(rng, 12, 32), dt=1.0 / 480,
                    steps=rng.randint(2, 6), every=rng.randint(1, 4), **block)
    # the sides of one tank lie within a factor of three of each other
    n = _log(rng, 20, 220)
    sides = [max(14, int(n * rng.uniform(0.34, 1.0))) for _ in range(2)] + [n]
    rng.shuffle(sides)
    big = max(sides)
    c = _frame("", sides, (0.0, 0.5, 0.6, 1.0), dt=1.0 / (480 if big < 100 else 960 if big < 200
                                                          else 1920),
               substeps=rng.randint(2, 6), mixed=rng.random() < 0.6,
               phases=rng.random() < 0.25, out="particles" if big < 72 else "grid")
    del c["name"]
    c.update(block)
    c["amg"] = not c["mixed"] and rng.random() < 0.4
    if big <= 140 and rng.random() < 0.2:
        c.update(cloth=2 * big + 1, y0=0.29, y1=0.29 + 0.6 * c["y1"], sigma=0.0)
    return c


# ---- inputs ----


def _box(c):
    """Cell size and the block's corners: the longest side is 1 m, the block is cut to whole
    cells of the tank (so that the seed moves the particles but not their number)."""
    n = (c["nx"], c["ny"], c["nz"])
    dx = 1.0 / max(n)
    y0 = min(int(c["y0"] / dx), int(0.6 * n[1]))
    top = [min(round(a / dx), m) for a, m in zip((c["x1"], c["y1"], c["z1"]), n)]
    top[1] = min(max(top[1], y0 + 4), n[1])
    return n, dx, (0.0, y0 * dx, 0.0), tuple(a * dx for a in top)


def _scene(c, seed):
    n, dx, lo, hi = _box(c)
    s = W.Scene(n, dx, precision=W.WC_MIXED if c.get("mixed") else W.WC_FP64)
    s.seed_block(lo, hi, seed=seed, sigma=c["sigma"])
    return s


def _uneven_liquid(c, seed):
    """A 7-point pressure system of a tank of liquid: walls below and on the sides (zero flux),
    an uneven free surface on top with the ghost-fluid 1/theta terms, DOFs numbered by 4x4x4
    bucket and then within it as the reference numbers them.  (rows, cols, values, rhs, cells)"""
    rng = np.random.default_rng(seed)
    nx, ny, nz = c["nx"], c["ny"], c["nz"]
    dims = (nx, ny, nz)
    x, z = np.arange(nx).reshape(nx, 1, 1), np.arange(nz).reshape(1, 1, nz)
    h = ny * (0.75 + 0.1 * np.sin(0.31 * x + 0.9) * np.cos(0.23 * z))
    j = np.arange(ny).reshape(1, ny, 1)
    liquid = np.broadcast_to(j, dims) < h
    i, jj, k = np.nonzero(liquid)
    bucket = ((k >> 2) * ((ny + 3) >> 2) + (jj >> 2)) * ((nx + 3) >> 2) + (i >> 2)
    order = np.argsort(bucket * 64 + (k & 3) * 16 + (jj & 3) * 4 + (i & 3), kind="stable")
    i, jj, k = i[order], jj[order], k[order]
    n = len(i)
    dof = np.full(dims, -1, dtype=np.int64)
    dof[i, jj, k] = np.arange(n)
    diag = np.zeros(n)
    rows, cols, vals = [], [], []
    for axis, d in enumerate(((1, 0, 0), (0, 1, 0), (0, 0, 1))):
        w = 0.7 + 0.6 * rng.random(dims)  # coefficient of the face above each cell on this axis
        theta = np.maximum(rng.random(dims), 0.01)
        for sign in (1, -1):
            # the neighbour's cell
            a, b, e = i + sign * d[0], jj + sign * d[1], k + sign * d[2]
            inside = (a >= 0) & (b >= 0) & (e >= 0) & (a < nx) & (b < ny) & (e < nz)
            other = np.full(n, -1, dtype=np.int64)
            other[inside] = dof[a[inside], b[inside], e[inside]]
            face = w[i, jj, k].copy()
            if sign < 0:
                face[inside] = w[a[inside], b[inside], e[inside]]
            wet = other >= 0
            diag[wet] += face[wet]
            rows.append(np.nonzero(wet)[0])
            cols.append(other[wet])
            vals.append(-face[wet])
            air = inside & ~wet
            diag[air] += face[air] / theta[i[air], jj[air], k[air]]
    rows.append(np.arange(n))
    cols.append(np.arange(n))
    vals.append(diag)
    rows, cols, vals = (np.concatenate(v) for v in (rows, cols, vals))
    o = np.lexsort((cols, rows))
    rows, cols, vals = rows[o], cols[o], vals[o]
    rs = np.zeros(n + 1, dtype=np.uint32)
    np.cumsum(np.bincount(rows, minlength=n), out=rs[1:])
    b = np.sin(0.11 * i + 0.07 * jj + 0.05 * k) + 0.3 * rng.standard_normal(n)
    return rs, cols.astype(np.uint32), vals, b, np.stack([i, jj, k], 1).astype(np.int32)


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind in ("pcg", "amgpcg"):
        return dict(case=c, system=_uneven_liquid(c, seed))
    s = _scene(c, seed)
    st = dict(case=c, scene=s)
    if kind == "exchange":
        st["host"] = s.particles_reference_layout()
    elif kind == "rollout":
        x, v, _ = s.particles()
        rng = np.random.default_rng(seed)
        st.update(x=x, v=v, target=x + 0.02 * rng.standard_normal((3, 1)))
    else:
        s.set_option("solver", 1 if c["amg"] else 0)
        if c["cloth"]:
            sheet = scenes.cloth_sheet(c["cloth"], 0.28, hi=(c["nx"] * s.dx, c["nz"] * s.dx),
                                       seed=seed)
            s.set_elasto(*scenes.elasto_args(sheet), prm=W.mix_params())
        if c["out"] == "particles":
            n = s.num_particles()
            st["arrays"] = [np.zeros((r, n)) for r in (3, 3, 9)]
        else:
            nn = s.grid_info()[1]
            st["arrays"] = [np.zeros(nn) for _ in range(3 if c["mixed"] else 4)]
    return st


# ---- one pass ----


def _substep(s, c):
    dt = c["dt"]
    if not c["phases"]:
        return s.substep(dt, TOL, MAXIT)[0]
    s.rebucketizeParticles()
    s.mapParticleNodesAPIC()
    s.stepVelocity(dt)
    ok = s.projectFine(dt, TOL, MAXIT)[0]
    s.applyPressureDragFluid(dt)
    s.map_node_particles_advect(dt)
    return ok


def _address(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_double))


def _read_back(st):
    """The frame's output into the program's arrays (the C interface's downloads)."""
    s, c, a = st["scene"], st["case"], st["arrays"]
    if c["out"] == "particles":
        status = W.lib().wc_get_particles_soa(s.h, *(_address(v) for v in a))
    else:
        status = 0
        for d, v in enumerate(a):
            name, axis = ("unew", d) if d < 3 else ("pressure", 0)
            status = status or W.lib().wc_download_field(s.h, W.FIELD[name], axis,
                                                         v.ctypes.data_as(ctypes.c_void_p))
    if status != W.WC_OK:
        raise W.WetclothError(W.lib().wc_last_error(s.h).decode())
    if c["mixed"]:
        return [torch.from_numpy(v).to(torch.float32) for v in a]
    return a


def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "pcg":
        rs, col, val, b, _ = state["system"]
        ok, x, _, _ = W.pcg_solve_csr(rs, col, val, b, tol=c["tol"], maxit=MAXIT)
        return dict(ok=ok, x=x)
    if kind == "amgpcg":
        rs, col, val, b, ijk = state["system"]
        ok, x, _, _ = W.amgpcg_solve_csr(rs, col, val, ijk, (c["nx"], c["ny"], c["nz"]), b,
                                         tol=c["tol"], maxit=MAXIT)
        return dict(ok=ok, x=x)
    s = state["scene"]
    if kind == "exchange":
        s.set_particles_reference_layout(*state["host"])
        ok = s.substep(c["dt"], TOL, MAXIT)[0]
        out = s.particles_reference_layout()
        if c["mixed"]:
            out = [torch.from_numpy(v).to(torch.float32) for v in out]
        return dict(ok=ok, state=list(out))
    if kind == "rollout":
        s.set_particles(state["x"], state["v"])
        ok, _ = s.rollout_forward(c["steps"], c["dt"], every=c["every"])
        x, v, C = s.particles()
        ok2, gx, gv, gC, gg = s.rollout_backward(c["dt"], 2.0 * (x - state["target"]))
        return dict(ok=ok and ok2, x=x, v=v, C=C, gx=gx, gv=gv, gC=gC, gg=gg)
    ok = True
    for _ in range(c["substeps"]):
        ok = _substep(s, c) and ok
    return dict(ok=ok, out=_read_back(state))


# ---- what a pass cannot do without, and the solves' exact answers ----


def work(case):
    """Algorithmic bytes and operations.  Per substep the particle state is read and written
    once and each liquid cell's grid values once; a MIC(0)-PCG iteration reads the matrix and
    the factor (4 values per row each) and touches its vectors 16 times per row, an AMG
    iteration about ten times that over all levels.  Iterations are those measured on the dam
    breaks: 125 at 256 cells, growing with the 3/4 power of the longest side; 6 with AMG."""
    c, kind = case, case["kind"]
    if kind in ("pcg", "amgpcg"):
        cells = 0.75 * c["nx"] * c["ny"] * c["nz"]
        big, amg = max(c["nx"], c["ny"], c["nz"]), kind == "amgpcg"
        iters = (12.0 if amg else 160.0 * (big / 256.0) ** 0.75)
        return dict(bytes=cells * (100.0 + iters * 8 * (240 if amg else 24)),
                    flops=cells * iters * (400 if amg else 40))
    n, dx, lo, hi = _box(c)
    cells = 1.0
    for a, b in zip(lo, hi):
        cells *= (b - a) / dx
    word = 4 if c.get("mixed") else 8
    amg = c.get("amg", False)
    iters = 6.0 if amg else 125.0 * (max(n) / 256.0) ** 0.75
    solve = cells * iters * word * (240 if amg else 24)
    sub = PPC * cells * 30 * word + cells * 200.0 + solve
    ops = PPC * cells * 4000.0 + cells * iters * (400 if amg else 40)
    if kind == "rollout":  # forward, replayed once more, and the adjoint of each substep
        return dict(bytes=3.0 * c["steps"] * sub, flops=3.0 * c["steps"] * ops)
    if kind == "exchange":
        return dict(bytes=sub + PPC * cells * 2 * 17 * 8, flops=ops)
    out = PPC * cells * 15 * 8 if c["out"] == "particles" else 4 * 8.0 * n[0] * n[1] * n[2]
    return dict(bytes=c["substeps"] * sub + out, flops=c["substeps"] * ops)


def exact(case, seed):
    """The solves' answers by conjugate gradients in FP64 with plain torch, to a residual far
    below theirs.  A substep's own outputs (a projection with its grids, boundary terms and
    transfers) have no short restatement apart from the library's."""
    if case["kind"] not in ("pcg", "amgpcg"):
        return None
    rs, col, val, b, _ = _uneven_liquid(case, seed)
    n = len(b)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    A = torch.sparse_csr_tensor(torch.from_numpy(rs.astype(np.int64)),
                                torch.from_numpy(col.astype(np.int64)), torch.from_numpy(val),
                                size=(n, n), device=dev)
    rows = np.repeat(np.arange(n), np.diff(rs.astype(np.int64)))
    inv = torch.from_numpy(1.0 / val[rows == col]).to(dev)
    r = torch.from_numpy(b).to(dev)
    x, z = torch.zeros_like(r), inv * r
    p, rho, stop = z.clone(), torch.dot(r, z), 1e-14 * r.abs().max()
    for it in range(20000):
        q = (A @ p.unsqueeze(1)).squeeze(1)
        alpha = rho / torch.dot(p, q)
        x += alpha * p
        r -= alpha * q
        if it % 10 == 9 and r.abs().max() <= stop:
            break
        z = inv * r
        new = torch.dot(r, z)
        p = z + (new / rho) * p
        rho = new
    return dict(ok=None, x=x)
