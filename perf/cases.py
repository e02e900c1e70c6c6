"""Timed cases of the particle-mesh library: what a program that uses it has it do.

Five kinds of call, each through the package's public entry points:

  loop     Simulation.run, the Landau / strong-field time loop on particles
           that stay on the GPU, in the FP32 and the FP64 state
  calls    one time step written with the reference's own calls on host
           arrays (push_x_, compute_rho, solve_, push_v_, push_x_)
  adjoint  Simulation.adjoint, the gradient of the field energy
  maxwell  Simulation.run_maxwell, the FDTD Vlasov-Maxwell loop
  ua       UASimulation.run, the uniformly accurate loop

listed() gives the cases, draw() more of the same ranges, prepare() the
inputs and handles a program holds before the call, run() one call and its
outputs, work() the bytes and operations it cannot do without, tolerance() the
difference another correct implementation may show, exact() the outputs in
64 bits from plain torch.
"""
import math

import numpy as np
import torch

from __graft_entry__ import load_package

DEV = "cuda"
F64 = torch.float64
KX = 0.5  # wave number of every perturbation; the domain is 4 pi long

STATES = {"f32": 1, "f64": 0}


# ------------------------------------------------------------------- cases

def listed():
    return [
        # The smallest calls: one step of the reference's example written with
        # its own functions on host arrays, on a test-sized mesh.
        {"name": "calls_cic_32x32_32768", "kind": "calls", "shape": "cic", "nx": 32, "ny": 32,
         "n": 32768, "dt": 0.1},
        # The reference README's Landau run: a small mesh, where launches and
        # latency count.
        {"name": "loop_cic_64x64_204800_f32", "kind": "loop", "shape": "cic", "state": "f32",
         "nx": 64, "ny": 64, "n": 204800, "dt": 0.1, "steps": 100, "sort": 8, "bz": "none",
         "alpha": 0.05, "tiles": 4},
        # The benchmark's headline: M6 Landau damping, FP32 state.
        {"name": "loop_m6_128x128_1e7_f32", "kind": "loop", "shape": "m6", "state": "f32",
         "nx": 128, "ny": 128, "n": 10_000_000, "dt": 0.05, "steps": 24, "sort": 12,
         "bz": "none", "alpha": 0.01, "tiles": 4},
        # The same in the FP64 state, the reference's arithmetic.
        {"name": "loop_m6_128x128_1e7_f64", "kind": "loop", "shape": "m6", "state": "f64",
         "nx": 128, "ny": 128, "n": 10_000_000, "dt": 0.05, "steps": 24, "sort": 12,
         "bz": "none", "alpha": 0.01, "tiles": 4},
        # Strong uniform magnetic field, CIC: the memory-bound pass.
        {"name": "loop_cic_256x256_1e8_f32", "kind": "loop", "shape": "cic", "state": "f32",
         "nx": 256, "ny": 256, "n": 100_000_000, "dt": 0.0125, "steps": 32, "sort": 32,
         "bz": "uniform", "alpha": 0.05, "tiles": 4},
        # The largest: M6 on 512 x 512, where particles cross cells quickly
        # and the sort is frequent.
        {"name": "loop_m6_512x512_2e8_f32", "kind": "loop", "shape": "m6", "state": "f32",
         "nx": 512, "ny": 512, "n": 200_000_000, "dt": 0.05, "steps": 8, "sort": 4,
         "bz": "none", "alpha": 0.05, "tiles": 2},
        # An ordinary run with nothing round about it: a mesh that is no power
        # of two, weighted particles, a magnetic field on the grid.
        {"name": "loop_tsc_100x75_300007_f64", "kind": "loop", "shape": "tsc", "state": "f64",
         "nx": 100, "ny": 75, "n": 300_007, "dt": 0.05, "steps": 40, "sort": 8, "bz": "grid",
         "alpha": 0.05, "tiles": 4, "weighted": True},
        # Gradients of the field energy, forward sweep and reverse sweep: the
        # FP32 state with CIC, and the FP64 state with M6.
        {"name": "adjoint_cic_128x128_2e6_f32", "kind": "adjoint", "shape": "cic",
         "state": "f32", "nx": 128, "ny": 128, "n": 2_000_000, "dt": 0.1, "steps": 40,
         "ckpt": 20, "sort": 4},
        {"name": "adjoint_m6_128x128_5e5_f64", "kind": "adjoint", "shape": "m6",
         "state": "f64", "nx": 128, "ny": 128, "n": 500_000, "dt": 0.05, "steps": 20,
         "ckpt": 10, "sort": 5},
        # The Vlasov-Maxwell loop of the reference's vm2d example, and on a
        # mesh that no longer fits one workgroup.
        {"name": "maxwell_128x16_204800", "kind": "maxwell", "nx": 128, "ny": 16, "n": 204_800,
         "dt": 0.01, "steps": 100},
        {"name": "maxwell_128x64_1024000", "kind": "maxwell", "nx": 128, "ny": 64,
         "n": 1_024_000, "dt": 0.01, "steps": 20},
        # The uniformly accurate loop of the reference's bupdate test.
        {"name": "ua_128x64_204800", "kind": "ua", "nx": 128, "ny": 64, "n": 204_800,
         "ntau": 16, "eps": 0.1, "dt": math.pi / 16, "steps": 2},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges."""
    kind = rng.choice(["loop", "loop", "loop", "calls", "adjoint", "maxwell", "ua"])
    if kind == "loop":
        state = rng.choice(["f32", "f32", "f64"])
        shape = rng.choice(["cic", "m6", "tsc", "m4"])
        if state == "f32":  # powers of two, as that state needs
            nx, ny = 2 ** rng.randint(5, 9), 2 ** rng.randint(5, 9)
        else:
            nx, ny = _log_int(rng, 24, 400), _log_int(rng, 24, 400)
            if rng.random() < 0.4:
                nx, ny = 2 ** rng.randint(5, 8), 2 ** rng.randint(5, 8)
        n = max(2 * nx * ny, _log_int(rng, 2e4, 2e7)) + rng.randint(0, 63)
        dt = rng.choice([0.0125, 0.05, 0.1])
        cell = 4 * math.pi / max(nx, ny)
        return {"kind": kind, "shape": shape, "state": state, "nx": nx, "ny": ny, "n": n,
                "dt": dt, "steps": rng.randint(9, 26),
                "sort": max(1, min(16, int(6.2 * cell / dt))),
                "bz": rng.choice(["none", "none", "uniform", "grid"]),
                "alpha": rng.choice([0.01, 0.05]), "tiles": 2 if max(nx, ny) > 256 else 4,
                "weighted": state == "f64" and rng.random() < 0.3}
    if kind == "calls":
        return {"kind": kind, "shape": rng.choice(["cic", "m6", "tsc", "m4"]),
                "nx": _log_int(rng, 24, 200), "ny": _log_int(rng, 24, 200),
                "n": _log_int(rng, 1e4, 5e5) + rng.randint(0, 63), "dt": 0.1}
    if kind == "adjoint":
        state = rng.choice(["f32", "f64"])
        side = [2 ** rng.randint(5, 8), 2 ** rng.randint(5, 8)]
        steps = rng.randint(8, 30)
        return {"kind": kind, "shape": rng.choice(["cic", "m6"]), "state": state,
                "nx": side[0], "ny": side[1],
                "n": max(4 * side[0] * side[1], _log_int(rng, 1e5, 6e5)) + rng.randint(0, 63),
                "dt": 0.05, "steps": steps, "ckpt": rng.randint(4, 12),
                "sort": max(1, min(6, int(3 * 4 * math.pi / max(side) / 0.05)))}
    if kind == "maxwell":
        nx, ny = _log_int(rng, 24, 200), _log_int(rng, 8, 100)
        return {"kind": kind, "nx": nx, "ny": ny,
                "n": max(4 * nx * ny, _log_int(rng, 5e4, 2e6)) + rng.randint(0, 63),
                "dt": 0.01, "steps": rng.randint(10, 40)}
    return {"kind": kind, "nx": _log_int(rng, 24, 160), "ny": _log_int(rng, 24, 160),
            "n": _log_int(rng, 2e4, 4e5) + rng.randint(0, 15), "ntau": rng.choice([8, 16, 32]),
            "eps": rng.choice([0.05, 0.1, 0.5]), "dt": math.pi / 16, "steps": 2}


def _lengths(case):
    if case["kind"] == "maxwell":
        return 2 * math.pi / KX, 1.0
    if case["kind"] == "ua":
        return 4 * math.pi, 2 * math.pi
    return 2 * math.pi / KX, 2 * math.pi / KX


# ------------------------------------------------------------------ inputs

def _rng(seed, salt=0):
    g = torch.Generator(device=DEV)
    g.manual_seed(1_000_003 * int(seed) + salt)
    return g


def _particles(case, seed):
    """(n, 5) rows x, y, vx, vy, w: density 1 + alpha cos(kx x), Maxwellian
    velocities.  The memory is that of a Fortran 5 x n array."""
    n = case["n"]
    lx, ly = _lengths(case)
    alpha = case.get("alpha", 0.05)
    g = _rng(seed)
    p = torch.empty((n, 5), dtype=F64, device=DEV)
    block = 1 << 24
    for a in range(0, n, block):
        b = min(n, a + block)
        u = torch.rand(b - a, dtype=F64, device=DEV, generator=g) * lx
        x = u.clone()  # invert u = x + (alpha / kx) sin(kx x)
        for _ in range(6):
            x -= (x + alpha / KX * torch.sin(KX * x) - u) / (1 + alpha * torch.cos(KX * x))
        p[a:b, 0] = x.clamp_(0.0, lx * (1 - 1e-15))
        p[a:b, 1] = torch.rand(b - a, dtype=F64, device=DEV, generator=g) * ly
        p[a:b, 2:4] = torch.randn((b - a, 2), dtype=F64, device=DEV, generator=g)
        w = lx * ly / n
        if case.get("weighted"):
            p[a:b, 4] = w * (0.5 + torch.rand(b - a, dtype=F64, device=DEV, generator=g))
        else:
            p[a:b, 4] = w
    return p


def _bz_grid(case):
    """A smooth magnetic field on the nodes, (nx, ny)."""
    i = np.arange(case["nx"]) / case["nx"]
    j = np.arange(case["ny"]) / case["ny"]
    return np.asfortranarray(1.0 + 0.3 * np.cos(2 * np.pi * i)[:, None]
                             * np.sin(2 * np.pi * j)[None, :])


def _bz(case):
    mode = case.get("bz", "none")
    return None if mode == "none" else 20.0 if mode == "uniform" else _bz_grid(case)


def _plasma(case, seed):
    """Positions (2, n) of density 1 + sin(y) + alpha cos(kx x) by rejection,
    and velocities of two drifting Maxwellians: the start of the UA loop."""
    n, alpha = case["n"], 0.05
    lx, ly = _lengths(case)
    rng = np.random.default_rng(seed)
    got, have = [], 0
    while have < n:
        x, y = rng.uniform(0, lx, n), rng.uniform(0, ly, n)
        z = (2.0 + alpha) * rng.uniform(size=n)
        keep = 1.0 + np.sin(y) + alpha * np.cos(KX * x) >= z
        got.append(np.stack([x[keep], y[keep]]))
        have += int(keep.sum())
    x = np.asfortranarray(np.concatenate(got, axis=1)[:, :n])
    v = rng.normal(size=(2, n))
    v[0] += 2.0 * rng.choice([-1.0, 1.0], n)
    return x, np.asfortranarray(v)


def _shape_of(pic, name):
    return {"cic": pic.CloudInCell, "m6": pic.M6, "tsc": pic.TriangularShapeCloud,
            "m4": pic.M4}[name]()


def _simulation(pic, case, seed):
    lx, ly = _lengths(case)
    mesh = pic.TwoDGrid(0.0, lx, case["nx"], 0.0, ly, case["ny"])
    p = _particles(case, seed)
    torch.cuda.synchronize()
    sim = pic.Simulation(mesh, None, _shape_of(pic, case.get("shape", "cic")))
    bz = _bz(case)
    if isinstance(bz, np.ndarray):
        sim.ctx.set_grid(pic._lib.PIC_GRID_BZ, bz)
        sim.ctx.set_bz(pic._lib.PIC_BZ_GRID)
    elif bz is not None:
        sim.ctx.set_bz(pic._lib.PIC_BZ_UNIFORM, bz)
    pic._lib.call("pic_set_particles_device", sim.ctx.h, p.data_ptr(), case["n"])
    sim.n = case["n"]
    sim.ctx.set_state(STATES[case.get("state", "f64")])
    sim.ctx.sync()
    del p
    torch.cuda.empty_cache()
    return mesh, sim


def prepare(case, seed):
    pic = load_package()
    state = {"case": case, "pic": pic}
    if case["kind"] == "calls":
        lx, ly = _lengths(case)
        state["mesh"] = pic.TwoDGrid(0.0, lx, case["nx"], 0.0, ly, case["ny"])
        state["group"] = pic.ParticleGroup(case["n"])
        state["group"].array[...] = _particles(case, seed).cpu().numpy().T
        state["poisson"] = pic.TwoDPoissonPeriodic(state["mesh"])
        state["kernel"] = _shape_of(pic, case["shape"])
        for k in ("ex", "ey", "bz"):
            state[k] = np.zeros((case["nx"], case["ny"]), order="F")
        return state
    if case["kind"] == "ua":
        lx, ly = _lengths(case)
        mesh = pic.TwoDGrid(0.0, lx, case["nx"], 0.0, ly, case["ny"])
        p = pic.Particles(case["n"], lx * ly / case["n"])
        p.x[...], p.v[...] = _plasma(case, seed)
        state["sim"] = pic.UASimulation(mesh, p, case["ntau"], case["eps"])
    else:
        state["mesh"], sim = _simulation(pic, case, seed)
        state["sim"] = sim
        if case["kind"] == "loop":
            sim.set_f32_tiles(case["tiles"])
        if case["kind"] == "maxwell":
            f = pic.FDTD(state["mesh"])
            x = np.linspace(0.0, state["mesh"].dimx, case["nx"] + 1)[:-1]
            f.ex[...] = (0.05 / KX * np.sin(KX * x))[:, None]
            sim.set_fdtd(f)
    if _returns_particles(case):
        state["particles"] = torch.empty((case["n"], 5), dtype=F64, device=DEV)
        torch.cuda.synchronize()
    return state


# --------------------------------------------------------------------- run

def _returns_particles(case):
    """The FP64 loops hand back their particles.  The FP32 loop's particles are
    left where they are: it re-sorts them by cell, so one offset that rounds
    the other way at a cell face reorders all that follow it, and two correct
    runs cannot be compared particle by particle.  Its fields and energies
    depend on every one of them."""
    return case["kind"] in ("maxwell", "ua") or (case["kind"] == "loop"
                                                 and case["state"] == "f64")


def _get_particles(s):
    ctx = s["sim"].ctx
    s["pic"]._lib.call("pic_get_particles_device", ctx.h, s["particles"].data_ptr())
    ctx.sync()
    return s["particles"]


def run(s):
    case, pic = s["case"], s["pic"]
    kind = case["kind"]
    if kind == "calls":
        p, mesh, kernel, dt = s["group"], s["mesh"], s["kernel"], case["dt"]
        pic.push_x_(p, mesh, 0.5 * dt)
        rho = pic.compute_rho(p, kernel, mesh)
        pic.solve_(s["ex"], s["ey"], s["poisson"], rho)
        pic.push_v_(p, kernel, mesh, s["ex"], s["ey"], s["bz"], dt)
        pic.push_x_(p, mesh, 0.5 * dt)
        return {"rho": rho, "ex": s["ex"], "ey": s["ey"], "particles": p.array}
    sim = s["sim"]
    if kind == "adjoint":
        energy, gx, gv = sim.adjoint(case["dt"], case["steps"], case["ckpt"], case["sort"])
        return {"energy": energy, "gx": gx, "gv": gv}
    if kind == "ua":
        out = {"energy": sim.run(case["dt"], case["steps"]), "e": sim.fields_e()}
    elif kind == "maxwell":
        out = {"energy": sim.run_maxwell(case["dt"], case["steps"])}
        f = sim.fdtd()
        out["ex"], out["ey"], out["bz"] = f.ex, f.ey, f.bz
    else:
        out = {"energy": sim.run(case["dt"], case["steps"], sort_every=case["sort"])}
        for k, which in (("rho", 0), ("ex", 1), ("ey", 2)):
            out[k] = sim.grid(which)
    if _returns_particles(case):
        out["particles"] = _get_particles(s)
    return out


# -------------------------------------------------------------------- work

# Operations a particle needs per step: two evaluations of the weights of a
# direction each, S^2 products, two gathered components, S^2 deposited sums.
_SIDE = {"cic": 2, "tsc": 4, "m4": 4, "m6": 6}
_WEIGHTS = {"cic": 2, "tsc": 16, "m4": 20, "m6": 40}


def _push_flops(shape, deposit=True):
    s = _SIDE[shape]
    return 2 * _WEIGHTS[shape] + 4 * s * s + 12 + (2 * _WEIGHTS[shape] + 2 * s * s if deposit else 0)


def work(case):
    """The particle state read once and written once per step (FP32 state: a
    cell and four floats; FP64 state: four doubles, and the weight where
    weights differ), the outputs, and the operations above."""
    n, kind, m = case["n"], case["kind"], case["nx"] * case["ny"]
    if kind == "calls":  # p.array in and out, the grids out
        return {"bytes": 80.0 * n + 24.0 * m, "flops": float(n) * _push_flops(case["shape"])}
    steps = case["steps"]
    if kind == "ua":
        # per sample and half step: about nine transforms along tau, the
        # gather, six sines
        per = case["ntau"] * (9 * 5 * math.log2(case["ntau"]) + 190 + 6 * 20)
        return {"bytes": 2.0 * steps * n * (64 + 64 * case["ntau"]) + 40.0 * n,
                "flops": 2.0 * steps * n * per}
    if kind == "maxwell":
        return {"bytes": 64.0 * n * steps + 40.0 * n, "flops": float(n) * steps * 90}
    f32 = case["state"] == "f32"
    state = 20 if f32 else 32 + (8 if case.get("weighted") else 0)
    if kind == "adjoint":
        # forward and recomputed step: state in and out; reverse: the state
        # and the adjoints in, the adjoints out
        adj = 16 if f32 else 32
        return {"bytes": float(n) * (steps * (4 * state + state + 2 * adj) + 32),
                "flops": 5.0 * n * steps * _push_flops(case["shape"])}
    wgt = 8 if case.get("weighted") else 0  # read only
    return {"bytes": float(n) * (steps * (2 * state - wgt)
                                 + (40 if _returns_particles(case) else 0)) + 24.0 * m,
            "flops": float(n) * steps * _push_flops(case["shape"])}


def tolerance(case):
    """From the distance to exact() and between runs whose sums are taken in
    another order (another sort interval).  FP64: loops up to 3e-13 from
    exact(), the rest below 2e-14.  FP32 loops: up to 8e-5 from exact(), 2e-6
    from one another; CIC adjoint 1.7e-3 from exact()."""
    kind = case["kind"]
    if kind == "adjoint" and case["state"] == "f32":
        # a CIC gradient jumps where a particle meets a cell face, so one
        # rounding of a position moves single entries by their own size
        return {"rel": 6e-3, "max": 0.99} if case["shape"] == "cic" else {"rel": 1e-4,
                                                                         "max": 1e-1}
    if kind == "loop":
        return {"rel": 1e-4, "max": 5e-3} if case["state"] == "f32" else {"rel": 5e-12,
                                                                         "max": 2e-10}
    return {"rel": 1e-12, "max": 5e-11}


# ------------------------------------------------- the same in 64 bits, torch

def _cell(x, d, n):
    xp = x / d
    f = torch.floor(xp.detach())
    return f.long() % n, xp - f


def _f_tsc(x):
    return torch.where(x <= 0.5, 0.75 - x * x,
                       torch.where(x <= 1.5, 0.5 * (1.5 - x) ** 2, torch.zeros_like(x)))


def _f_m4(x):
    near = 1 - 1.5 * x * x + 0.75 * x ** 3
    far = 0.25 * (2 - x) ** 3
    return torch.where(x >= 1, torch.where(x > 2, torch.zeros_like(x), far), near) * 2 / 3


def _m6(t):
    def p3(u):
        return ((((10 * u - 20) * u - 20) * u + 20) * u + 50) * u + 26

    def p4(u):
        return ((((-5 * u + 5) * u + 10) * u + 10) * u + 5) * u + 1

    s = 1 - t
    return [s ** 5 / 120, p4(s) / 120, p3(s) / 120, p3(t) / 120, p4(t) / 120, t ** 5 / 120]


def _weights(shape, d, deposit):
    """(offset of the first node, weights) of a direction."""
    if shape == "cic":
        return 0, [1 - d, d]
    if shape == "m6":
        return -2, _m6(d)
    f = _f_tsc if shape == "tsc" and deposit else _f_m4
    return -1, [f(1 + d), f(d), f(1 - d), f(2 - d)]


def _stencil(case, x, y, deposit):
    """Yields (node index j nx + i, weight) over the stencil."""
    nx, ny = case["nx"], case["ny"]
    lx, ly = _lengths(case)
    i, fx = _cell(x, lx / nx, nx)
    j, fy = _cell(y, ly / ny, ny)
    o, wx = _weights(case.get("shape", "cic"), fx, deposit)
    _, wy = _weights(case.get("shape", "cic"), fy, deposit)
    for v, b in enumerate(wy):
        row = (j + (o + v)) % ny * nx
        for u, a in enumerate(wx):
            yield row + (i + (o + u)) % nx, a * b


_BLOCK = 1 << 24


def _blocks(n):
    return [slice(a, min(n, a + _BLOCK)) for a in range(0, n, _BLOCK)]


def _deposit(case, x, y, w):
    acc = torch.zeros(case["nx"] * case["ny"], dtype=F64, device=DEV)
    for b in _blocks(case["n"]):
        wb = w[b] if w.dim() else w
        for q, a in _stencil(case, x[b], y[b], True):
            acc = acc.index_add(0, q, a * wb)
    lx, ly = _lengths(case)
    return acc / (lx / case["nx"] * ly / case["ny"])


def _solve(case, rho):
    """(ex, ey) as flat node arrays, x fastest."""
    nx, ny = case["nx"], case["ny"]
    lx, ly = _lengths(case)
    r = torch.fft.rfft2(rho.reshape(ny, nx))
    kx = (2 * math.pi / lx) * torch.arange(nx // 2 + 1, dtype=F64, device=DEV)[None, :]
    j = torch.arange(ny, dtype=F64, device=DEV)
    ky = ((2 * math.pi / ly) * torch.where(j < ny // 2, j, j - ny))[:, None]
    k2 = kx * kx + ky * ky
    k2[0, 0] = 1.0
    ex = torch.fft.irfft2(-1j * kx / k2 * r, s=(ny, nx))
    ey = torch.fft.irfft2(-1j * ky / k2 * r, s=(ny, nx))
    return ex.reshape(-1), ey.reshape(-1)


def _kick(case, x, y, vx, vy, ex, ey, bz, dt):
    e1 = e2 = b3 = 0.0
    for q, a in _stencil(case, x, y, False):
        e1 = e1 + a * ex.index_select(0, q)
        e2 = e2 + a * ey.index_select(0, q)
        if isinstance(bz, torch.Tensor):
            b3 = b3 + a * bz.index_select(0, q)
    if isinstance(bz, float):
        b3 = bz
    vx, vy = vx + 0.5 * dt * e1, vy + 0.5 * dt * e2
    if bz is not None:
        t = 0.5 * dt * b3
        s = 2 * t / (1 + t * t)
        vx = vx + vy * t
        vy = vy - vx * s
        vx = vx + vy * t
    return vx + 0.5 * dt * e1, vy + 0.5 * dt * e2


def _wrap(x, l):
    x = torch.where(x > l, x - l, x)
    return torch.where(x < 0, x + l, x)


def _grid(case, g):
    return g.reshape(case["ny"], case["nx"]).T


def _exact_loop(case, seed):
    side = _SIDE[case["shape"]]
    if case["n"] * case["steps"] * side * side > 2.5e10:
        return None  # too long
    p = _particles(case, seed)
    x, y, vx, vy, w = (p[:, k].clone() for k in range(5))
    del p
    lx, ly = _lengths(case)
    h = 0.5 * case["dt"]
    bz = _bz(case)
    if isinstance(bz, np.ndarray):
        bz = torch.from_numpy(np.ascontiguousarray(bz.T)).reshape(-1).to(DEV)
    x, y = _wrap(x + h * vx, lx), _wrap(y + h * vy, ly)
    energy = []
    cell = lx / case["nx"] * ly / case["ny"]
    for s in range(case["steps"]):
        rho = _deposit(case, x, y, w)
        ex, ey = _solve(case, rho)
        energy.append([float((ex * ex).sum() * cell), float((ey * ey).sum() * cell)])
        for b in _blocks(case["n"]):
            vx[b], vy[b] = _kick(case, x[b], y[b], vx[b], vy[b], ex, ey, bz, case["dt"])
        for _ in range(1 if s == case["steps"] - 1 else 2):
            x, y = _wrap(x + h * vx, lx), _wrap(y + h * vy, ly)
    out = {"energy": np.array(energy), "rho": _grid(case, rho - rho.mean()),
           "ex": _grid(case, ex), "ey": _grid(case, ey)}
    if _returns_particles(case):
        out["particles"] = None  # in the order of the last sort
    return out


def _exact_calls(case, seed):
    p = _particles(case, seed)
    x, y, vx, vy, w = (p[:, k].clone() for k in range(5))
    lx, ly = _lengths(case)
    h = 0.5 * case["dt"]
    x, y = _wrap(x + h * vx, lx), _wrap(y + h * vy, ly)
    rho = _deposit(case, x, y, w)
    rho = rho - rho.mean()
    ex, ey = _solve(case, rho)
    vx, vy = _kick(case, x, y, vx, vy, ex, ey, None, case["dt"])
    x, y = _wrap(x + h * vx, lx), _wrap(y + h * vy, ly)
    return {"rho": _grid(case, rho), "ex": _grid(case, ex), "ey": _grid(case, ey),
            "particles": torch.stack([x, y, vx, vy, w])}


def _exact_adjoint(case, seed):
    side = _SIDE[case["shape"]]
    if case["n"] * case["steps"] * side * side * 40 > 4e10:
        return None  # the tape would be too large
    p = _particles(case, seed)
    x0, y0, u0, v0 = (p[:, k].clone().requires_grad_() for k in range(4))
    w = p[0, 4].clone()
    lx, ly = _lengths(case)
    h = 0.5 * case["dt"]
    x, y, vx, vy = x0 + h * u0, y0 + h * v0, u0, v0
    cell = lx / case["nx"] * ly / case["ny"]
    for s in range(case["steps"]):
        ex, ey = _solve(case, _deposit(case, x, y, w))
        if s == case["steps"] - 1:
            break
        vx, vy = _kick(case, x, y, vx, vy, ex, ey, None, case["dt"])
        x, y = x + case["dt"] * vx, y + case["dt"] * vy
    energy = (ex * ex + ey * ey).sum() * cell
    g = torch.autograd.grad(energy, [x0, y0, u0, v0])
    return {"energy": float(energy.detach()), "gx": torch.stack(g[:2]), "gv": torch.stack(g[2:])}


def _exact_maxwell(case, seed):
    nx, ny, dt = case["nx"], case["ny"], case["dt"]
    lx, ly = _lengths(case)
    dx, dy = lx / nx, ly / ny
    p = _particles(case, seed)
    x, y, vx, vy, w = (p[:, k].clone() for k in range(5))
    i = torch.arange(nx, dtype=F64, device=DEV)
    # fields as (ny, nx): the Yee fields and their periodic images
    ex = (0.05 / KX * torch.sin(KX * i * dx))[None, :].expand(ny, nx).clone()
    ey, bz = torch.zeros_like(ex), torch.zeros_like(ex)

    def ahead(f, d):
        return torch.roll(f, -1, d)

    def back(f, d):
        return torch.roll(f, 1, d)

    def faraday(b, step):
        return b + step * ((ahead(ex, 0) - ex) / dy - (ahead(ey, 1) - ey) / dx)

    energy = []
    for s in range(case["steps"]):
        if s:
            bz = faraday(bz, 0.5 * dt)
        nex, ney = 0.5 * (back(ex, 1) + ex), 0.5 * (back(ey, 0) + ey)
        nbz = 0.25 * (back(back(bz, 0), 1) + back(bz, 0) + back(bz, 1) + bz)
        vx, vy = _kick(case, x, y, vx, vy, nex.reshape(-1), ney.reshape(-1), nbz.reshape(-1), dt)
        x, y = _wrap(x + 0.5 * dt * vx, lx), _wrap(y + 0.5 * dt * vy, ly)
        jx = torch.zeros(nx * ny, dtype=F64, device=DEV)
        jy = torch.zeros_like(jx)
        for q, a in _stencil(case, x, y, True):
            jx.index_add_(0, q, a * vx * w / (dx * dy))
            jy.index_add_(0, q, a * vy * w / (dx * dy))
        jx, jy = jx.reshape(ny, nx), jy.reshape(ny, nx)
        x, y = _wrap(x + 0.5 * dt * vx, lx), _wrap(y + 0.5 * dt * vy, ly)
        bz = faraday(bz, 0.5 * dt)
        ex = ex + dt * (bz - back(bz, 0)) / dy - dt * 0.5 * (jx + ahead(jx, 1))
        ey = ey - (dt * (bz - back(bz, 1)) / dx - dt * 0.5 * (jy + ahead(jy, 0)))
        total = (ex * ex).sum() + (ex[0] * ex[0]).sum()  # the ghost row counts too
        energy.append(0.5 * math.log(float(total) * dx * dy))
    return {"energy": np.array(energy), "ex": torch.cat([ex, ex[:1]]).T,
            "ey": torch.cat([ey, ey[:, :1]], 1).T, "bz": bz.T,
            "particles": torch.stack([x, y, vx, vy, w], 1)}


def _m6_nodes(case, x, y, shift):
    """Nodes and weights of the M6 stencil at positions in the domain; shift:
    the node offsets of compute_rho_m6!(fields, particles), one node low but
    for the particle's own."""
    nx, ny = case["nx"], case["ny"]
    lx, ly = _lengths(case)
    px, py = x / (lx / nx), y / (ly / ny)
    i, j = torch.trunc(px), torch.trunc(py)
    wx, wy = _m6(px - i), _m6(py - j)
    off = [-3, -2, 0, 0, 1, 2] if shift else [-2, -1, 0, 1, 2, 3]
    for a in range(6):
        ia = (i.long() + off[a]) % nx
        for b in range(6):
            yield (j.long() + off[b]) % ny * nx + ia, wx[a] * wy[b]


def _m6_rho(case, x, y, w, shift):
    lx, ly = _lengths(case)
    acc = torch.zeros(case["nx"] * case["ny"], dtype=F64, device=DEV)
    for q, a in _m6_nodes(case, x, y, shift):
        acc.index_add_(0, q, a * w)
    return acc / (lx / case["nx"] * ly / case["ny"])


def _m6_gather(case, x, y, ex, ey):
    lx, ly = _lengths(case)
    e1, e2 = torch.zeros_like(x), torch.zeros_like(x)
    for q, a in _m6_nodes(case, x.remainder(lx), y.remainder(ly), False):
        e1 += a * ex[q]
        e2 += a * ey[q]
    return e1, e2


def _exact_ua(case, seed):
    """The loop of the UA scheme: per particle ntau samples in the fast
    variable, prediction and correction."""
    nt, eps, dt, n = case["ntau"], case["eps"], case["dt"], case["n"]
    lx, ly = _lengths(case)
    cell = lx / case["nx"] * ly / case["ny"]
    x, v = (torch.from_numpy(np.ascontiguousarray(a)).to(DEV) for a in _plasma(case, seed))
    w = lx * ly / n
    # the prologue: the deposit puts the particles at x mod the domain
    x = torch.stack([x[0].remainder(lx), x[1].remainder(ly)])
    ex, ey = _solve(case, _m6_rho(case, x[0], x[1], w, True))
    pe = torch.stack(_m6_gather(case, x[0], x[1], ex, ey))
    l = torch.fft.fftfreq(nt, 1.0 / nt, dtype=F64, device=DEV)[:, None]
    tau = (torch.arange(nt, dtype=F64, device=DEV) * (2 * math.pi / nt))[:, None]
    c, s = torch.cos(tau), torch.sin(tau)
    l1 = torch.where(l == 0, torch.ones_like(l), l)
    fft, ifft = (lambda z: torch.fft.fft(z, dim=-2)), (lambda z: torch.fft.ifft(z, dim=-2))
    energies = np.zeros((2, case["steps"]))

    def b_of(a, b):
        return 1 + 0.5 * torch.sin(a) * torch.sin(b)

    def force(xr, yt, b, e1, e2):
        d = (b_of(xr[0], xr[1]) - b) / eps
        fx = torch.stack([(c * yt[0] + s * yt[1]) / b, (-s * yt[0] + c * yt[1]) / b])
        t1 = e1 + d * (c * yt[1] - s * yt[0])
        t2 = e2 + d * (-c * yt[0] - s * yt[1])
        fy = torch.stack([(c * t1 - s * t2) / b, (s * t1 + c * t2) / b])
        return fft(fx), fft(fy)

    def solve(half, step):
        ex, ey = _solve(case, _m6_rho(case, x[0], x[1], w, False))
        gx, gy = _grid(case, ex), _grid(case, ey)
        q = (gx * gx + gy * gy)
        q = q.sum() + q[0].sum() + q[:, 0].sum() + q[0, 0]
        energies[half, step] = float(q) * cell
        return ex, ey

    for step in range(case["steps"]):
        b = b_of(x[0], x[1])
        t = dt * b
        vb = v / b
        h1, h2 = eps * (s * vb[0] - c * vb[1]), eps * (s * vb[1] + c * vb[0])
        xt = torch.stack([x[0] + h1 + eps * vb[1], x[1] + h2 - eps * vb[0]])
        d = (b_of(xt[0], xt[1]) - b) / eps
        eb1 = ((c * v[1] - s * v[0]) * d + pe[0]) / b
        eb2 = ((-c * v[0] - s * v[1]) * d + pe[1]) / b
        r = fft(torch.stack([c * eb1 - s * eb2, s * eb1 + c * eb2]).to(torch.complex128))
        r = ifft(torch.where(l == 0, r, -1j * r / l1))
        yt = v[:, None, :] + eps * (r - r[:, :1, :])
        elt = torch.exp(-1j * l * t / eps)
        pl = torch.where(l == 0, t.to(torch.complex128), eps * 1j * (elt - 1) / l1)
        ql = torch.where(l == 0, (t * t / 2).to(torch.complex128),
                         eps * (eps * (1 - elt) - 1j * l * t) / l1 ** 2)

        def place(spectrum):
            """x(t) from the tau-spectrum of the samples, into the domain."""
            pos = (spectrum * (torch.conj(elt) / nt)).sum(-2).real
            return torch.stack([pos[0].remainder(lx), pos[1].remainder(ly)])

        e1, e2 = _m6_gather(case, xt[0], xt[1], ex, ey)
        fx, fy = force(xt, yt, b, e1, e2)
        xs, ys = fft(xt.to(torch.complex128)), fft(yt)
        xp, yp = elt * xs + pl * fx, elt * ys + pl * fy
        x = place(xp)
        ex, ey = solve(0, step)
        xq, yq = ifft(xp), ifft(yp)
        e1, e2 = _m6_gather(case, xq.real[0], xq.real[1], ex, ey)
        gx, gy = force(xq.real, yq, b, e1, e2)
        xp, yp = xp + ql * (gx - fx) / t, yp + ql * (gy - fy) / t
        x = place(xp)
        q = (yp / nt * torch.conj(elt)).sum(-2).real
        ct, st = torch.cos(t / eps), torch.sin(t / eps)
        v = torch.stack([ct * q[0] + st * q[1], ct * q[1] - st * q[0]])
        ex, ey = solve(1, step)

    def ghost(g):
        g = _grid(case, g)
        g = torch.cat([g, g[:1]], 0)
        return torch.cat([g, g[:, :1]], 1)

    return {"energy": energies, "e": torch.stack([ghost(ex), ghost(ey)]),
            "particles": torch.stack([x[0], x[1], v[0], v[1], torch.full_like(x[0], w)], 1)}


def exact(case, seed):
    return {"loop": _exact_loop, "calls": _exact_calls, "adjoint": _exact_adjoint,
            "maxwell": _exact_maxwell, "ua": _exact_ua}[case["kind"]](case, seed)
