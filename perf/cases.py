"""Performance cases of the plasma step: what users of the package run.

A pass is 20 steps, the sort cadence of the shipped configurations, so that
every pass after the first holds one cell sort and the inflows that fall due:
`Simulation.step`, `Simulation2D.step`, the same 3D loop driven routine by
routine, or one forward and backward sweep of the adjoint.

The outputs of a stepping pass are the state that the simulation keeps on the
GPU.  Its planes can be had through `download_field` only, a copy to the host
that a program makes when it writes a field dump every few hundred steps and
not after each pass; `State` therefore names them and copies a plane when it
is looked at.  Nothing that the steps compute is left for that moment.

`exact` restates the steps in plain torch with 64-bit numbers: counter-based
loading and inflow, gather, push, deposit, fields, the Poisson corrections
and, through autograd, the gradient of the adjoint's loss.
"""
import math

import numpy as np
import torch

import plasmasim_amd as ps

STEPS = 20
PLANES = ("ex", "ey", "ez", "bx", "by", "bz", "jix", "jiy", "jiz", "jex", "jey", "jez",
          "ni", "ne")


# ---------------------------------------------------------------------------
# the cases


def case3d(name, kind, nx, ny, nz, ppc, precision, tile, **more):
    c = {"name": name, "kind": kind, "nx": nx, "ny": ny, "nz": nz, "ppc": ppc,
         "precision": precision, "tx": tile[0], "ty": tile[1], "tz": tile[2],
         "deterministic": False, "thrust": False, "poisson_every": 0, "mass": 100.0,
         "drift": 0.1, "steps": STEPS}
    c.update(more)
    return c


def case2d(name, nx, nz, ppc, precision, tile, **more):
    c = {"name": name, "kind": "step2d", "nx": nx, "nz": nz, "ppc": ppc,
         "precision": precision, "tx": tile, "tz": tile, "poisson_every": 1,
         "inflow_every": 50, "steps": STEPS}
    c.update(more)
    return c


def listed():
    return [
        # the smallest shipped grid: a smoke run, bound by launches
        case3d("tiny_fp64", "step3d", 8, 8, 16, 4, "fp64", (0, 0, 0)),
        # the shipped parity run, particles in the reference's order
        case3d("cube32_fp64", "step3d", 32, 32, 32, 16, "fp64", (0, 0, 0)),
        # an exploratory run on a grid that no tile size divides
        case3d("odd_fp32", "step3d", 31, 27, 45, 8, "fp32", (0, 0, 0), thrust=True),
        # a desktop-size production run with the force record of every step
        case3d("cube64_fp32", "step3d", 64, 64, 64, 32, "fp32", (4, 4, 8), thrust=True),
        # a reproducible run (fixed summation order), heavy ions, ragged grid
        case3d("ragged_det_fp32", "step3d", 60, 44, 100, 27, "fp32", (4, 4, 4),
               deterministic=True, mass=400.0, drift=0.05),
        # the headline workload, in both numeric forms
        case3d("cube128_fp32", "step3d", 128, 128, 128, 64, "fp32", (8, 4, 4), thrust=True),
        case3d("cube128_fp64", "step3d", 128, 128, 128, 64, "fp64", (8, 4, 4), thrust=True),
        # a host program that keeps its own loop and calls one routine after
        # the other, with the diagnostics line that it prints now and then
        case3d("loop48_fp32", "loop3d", 48, 48, 96, 32, "fp32", (4, 4, 8)),
        # the 2D3V step: small, the full workload, and the plain form
        case2d("plane256_fp32", 256, 256, 16, "fp32", 16),
        case2d("plane2048_fp32", 2048, 2048, 100, "fp32", 16, inflow_every=250),
        case2d("plane512_fp64", 512, 512, 36, "fp64", 16),
        # gradient of the thrust over a short window
        case3d("adjoint64_fp32", "adjoint", 64, 64, 64, 32, "fp32", (4, 4, 8), window=10,
               radius=10.0, points=256),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _size(rng, lo, hi, tile):
    """A size of about `lo`..`hi` cells that `tile` divides."""
    return max(-(-lo // tile), round(_log(rng, lo, hi) / tile)) * tile


# tile shapes whose window of sums fits the pass (as the shipped ones do)
TILES = ((4, 4, 8), (8, 4, 4), (4, 4, 4), (3, 4, 5), (5, 5, 5), (6, 3, 4), (4, 4, 7))


def draw(rng):
    kind = rng.choice(("step3d",) * 6 + ("step2d",) * 3 + ("loop3d", "adjoint"))
    precision = rng.choice(("fp32", "fp32", "fp64"))
    if kind == "step2d":
        if rng.random() < 0.5:  # the Poisson correction takes powers of two
            nx, nz = (1 << rng.randint(5, 10) for _ in range(2))
            tile, poisson = rng.choice((8, 16)), 1
        else:
            tile, poisson = rng.choice((9, 12, 15)), 0
            nx, nz = (tile * max(3, round(_log(rng, 32, 900) / tile)) for _ in range(2))
        ppc = max(2, min(100, int(_log(rng, 4, 120)), int(3e7 / (nx * nz))))
        c = case2d("", nx, nz, ppc, precision, tile, poisson_every=poisson,
                   inflow_every=rng.choice((5, 50)))
    else:
        big = 24 if kind == "adjoint" else 40 if kind == "loop3d" else 100
        tile = list(rng.choice(TILES))
        n = [_size(rng, lo, big, t) for lo, t in zip((8, 8, 16), tile)]
        cells = n[0] * n[1] * n[2]
        ppc = max(2, min(64, int(_log(rng, 3, 80)), int(3e7 / cells)))
        if kind == "step3d" and cells * ppc < 300000 and rng.random() < 0.3:
            tile = [0, 0, 0]
        more = {"mass": rng.choice((25.0, 100.0, 400.0)), "drift": rng.choice((0.05, 0.1))}
        if kind == "step3d":
            more["thrust"] = rng.random() < 0.5
            more["deterministic"] = precision == "fp32" and rng.random() < 0.25
            if all(s & (s - 1) == 0 for s in n):
                more["poisson_every"] = rng.choice((0, 1))
        if kind == "adjoint":
            more.update(window=5, radius=float(min(3, min(n) // 2 - 2)), points=64, steps=10)
        c = case3d("", kind, n[0], n[1], n[2], ppc, precision, tile, **more)
    del c["name"]
    return c


# ---------------------------------------------------------------------------
# what a program has in hand before the pass


def config(case, seed):
    fp64 = case["precision"] == "fp64"
    if case["kind"] == "step2d":
        c = ps.preset2d(3)
        nx, nz = case["nx"], case["nz"]
        n0 = c.weight[0] * c.ppc
        c.nx, c.nz, c.ppc = nx, nz, case["ppc"]
        c.weight[0] = c.weight[1] = n0 / case["ppc"]
        c.tile[0], c.tile[1] = case["tx"], case["tz"]
        c.poisson_every, c.inflow_every = case["poisson_every"], case["inflow_every"]
        layer, margin = (32, 16) if nz >= 1024 else (max(nz // 16, 4), max(nz // 32, 4))
        c.absorb[1] = layer
        c.ballistic_lo[1], c.ballistic_hi[1] = margin * c.dx, (nz + 4 - margin) * c.dx
        c.phi_lo[0], c.phi_hi[0] = 2, nx + 2
        c.phi_lo[1], c.phi_hi[1] = layer, nz + 4 - layer
        c.ext_k = (nx + 4) // 2 + 1
        c.ext_m[0], c.ext_m[1] = (nz + 4) // 2 - 3, (nz + 4) // 2 + 2
        c.ext_ramp = 1000 if nz >= 1024 else 200
        standoff = min(64.0, nz / 16.0)
        c.ext_current = math.sqrt(standoff ** 4 * math.pi ** 2 * n0 * c.mass[0]
                                  * c.vdrift ** 2 / (c.mu0 * 4.0 * 2.5 ** 2))
    else:
        c = ps.preset(4)
        n0 = c.weight[0] * c.ppc
        c.nx, c.ny, c.nz, c.ppc = case["nx"], case["ny"], case["nz"], case["ppc"]
        c.weight[0] = c.weight[1] = n0 / case["ppc"]
        c.mass[0], c.vdrift[2] = case["mass"], case["drift"]
        standoff = max(3.0, min(c.nx, c.ny, c.nz) / 4.0)
        c.dipole_m = math.sqrt(standoff ** 6 * 8.0 * math.pi ** 2 * n0 * c.mass[0]
                               * c.vdrift[2] ** 2 / c.mu0)
        layer = max(c.nz // 8, 2)
        c.absorb[2] = layer
        c.ballistic_lo[2], c.ballistic_hi[2] = 2.0 + layer + 2, c.nz + 2.0 - layer - 2
        c.tile[0], c.tile[1], c.tile[2] = case["tx"], case["ty"], case["tz"]
        c.poisson_every, c.phi_margin = case["poisson_every"], layer + 2
        if case["deterministic"]:
            c.deposit = ps.PIC_DEPOSIT_DETERMINISTIC
    if case["kind"] == "adjoint":  # injected particles are appended, not refilled
        slabs = 4 * c.nx * c.ny * c.ppc
        c.capacity = (c.nx * c.ny * c.nz * c.ppc
                      + slabs * (2 + case["steps"] // c.inflow_every) + 4096)
    c.precision = ps.PIC_FP64 if fp64 else ps.PIC_FP32
    c.seed = 1000 + seed
    return c


def prepare(case, seed):
    c = config(case, seed)
    if case["kind"] == "step2d":
        sim = ps.Simulation2D(c)
    else:
        sim = ps.Simulation(c)
    if case["kind"] == "adjoint":
        return {"case": case, "sim": sim, "p": parameters(case, seed, c)}
    sim.load_particles()
    sim.begin()
    if case.get("thrust"):
        sim.thrust_ave(True)
    sim.sync()
    return {"case": case, "sim": sim, "c_add": 0, "c_sort": 0}


def parameters(case, seed, c):
    """(Mx, My, Mz, V) of one gradient: the moment a few degrees off its axis."""
    r = np.random.default_rng(seed)
    t = r.uniform(-0.1, 0.1, 2)
    m = c.dipole_m * np.array([math.sin(t[0]), math.cos(t[0]) * math.cos(t[1]),
                               math.cos(t[0]) * math.sin(t[1])])
    return np.array([*m, c.vdrift[2]])


class State(dict):
    """The simulation's planes, particle counts and force record by name; an
    entry is copied to the host when it is read."""

    def __init__(self, sim, thrust):
        super().__init__({k: None for k in PLANES + ("particles",)})
        if thrust:
            self["thrust"] = None
        self.sim = sim

    def __getitem__(self, k):
        if k == "particles":
            return np.array([float(self.sim.particle_count(s)) for s in (0, 1)])
        if k == "thrust":
            return self.sim.thrust_ave_get()[0]
        return self.sim.download_field(k)


def run(state):
    case, sim = state["case"], state["sim"]
    if case["kind"] == "adjoint":
        loss = sim.adj_forward(state["p"], case["steps"], case["window"], case["radius"],
                               case["points"])
        return {"loss": loss, "grad": sim.adj_backward()}
    if case["kind"] == "loop3d":
        every = sim.cfg
        for _ in range(case["steps"]):
            sim.renew_grid()
            if state["c_sort"] > every.sort_every - 1:
                state["c_sort"] = 0
                sim.sort(0)
                sim.sort(1)
            if state["c_add"] > every.inflow_every - 1:
                state["c_add"] = 0
                sim.inflow()
            sim.renew_b_half()
            sim.halo_b()
            sim.push_deposit_j(0)
            sim.push_deposit_j(1)
            sim.renew_b_half()
            sim.halo_b()
            sim.drift_deposit_n(0)
            sim.drift_deposit_n(1)
            sim.fold_current()
            sim.renew_e()
            sim.halo_e()
            sim.particle_boundary()
            state["c_sort"] += 1
            state["c_add"] += 1
        sim.diagnose()  # the line that the program prints
        return State(sim, False)
    sim.step(case["steps"])
    return State(sim, bool(case.get("thrust")))


def work(case):
    """Each step reads and writes every particle and every field value once:
    the particle state of the numeric form, E and B (old and new, in two half
    steps), the currents and the densities.  The adjoint runs the steps twice
    and reads and writes the particle adjoints (6 doubles) once per step."""
    cells = case["nx"] * case.get("ny", 1) * case["nz"]
    n = 2 * cells * case["ppc"]
    fp64 = case["precision"] == "fp64"
    if case["kind"] == "step2d":
        per_particle, per_cell, flops = (80, 240, 200) if fp64 else (48, 120, 200)
    else:
        per_particle, per_cell, flops = (96, 448, 350) if fp64 else (56, 224, 350)
    b = case["steps"] * (n * per_particle + cells * per_cell)
    f = case["steps"] * n * flops
    if case["kind"] == "adjoint":
        b = 2 * b + case["steps"] * (n * 96 + cells * 18 * 16)
        f = 4 * f
    return {"bytes": float(b), "flops": float(f)}


def tolerance(case):
    """About four times the distance from `exact` after the pass's steps.  fp32
    in 3D: planes up to 2.7e-5, single nodes next to the dipole up to 1e-2 of
    the plane's rms (electrons there part quickly); in 2D 1.7e-6 and 1.5e-4;
    the adjoint's loss 7.9e-7.  fp64: 4e-14, two runs (sums in another order)
    2e-13 apart and single nodes 5e-11."""
    fp64 = case["precision"] == "fp64"
    if case["kind"] == "adjoint":
        return {"rel": 1e-9 if fp64 else 4e-6}
    if fp64:
        return {"rel": 1e-12, "max": 2e-10}
    if case["kind"] == "step2d":
        return {"rel": 8e-6, "max": 6e-4}
    return {"rel": 1.2e-4, "max": 0.04}


# ---------------------------------------------------------------------------
# the same steps in plain torch, 64 bits

CHUNK = 1 << 21  # particles handled at a time
DEV = torch.device("cuda" if torch.cuda.is_available() else "cpu")
F8 = torch.float64


def philox(c, k0, k1):
    """Philox4x32-10 (Salmon et al., SC'11) of four int64 tensors of 32 bits."""
    m32 = 0xFFFFFFFF
    c0, c1, c2, c3 = c
    for _ in range(10):
        p0, p1 = c0 * 0xD2511F53, c2 * 0xCD9E8D57
        c0, c1, c2, c3 = (((p1 >> 32) & m32) ^ c1 ^ k0, p1 & m32,
                          ((p0 >> 32) & m32) ^ c3 ^ k1, p0 & m32)
        k0, k1 = (k0 + 0x9E3779B9) & m32, (k1 + 0xBB67AE85) & m32
    return c0, c1, c2, c3


def drawn(seed, sp, event, idx):
    """Three position fractions and three normals of the particles `idx`."""
    one = torch.ones_like(idx)
    w = [philox((idx & 0xFFFFFFFF, idx >> 32, one * event, one * (4 * sp + d)),
                seed & 0xFFFFFFFF, seed >> 32) for d in range(4)]

    def u(d, j):
        return ((w[d][j] >> 5).to(F8) * 67108864.0 + (w[d][j + 1] >> 6).to(F8)) / 9007199254740992.0

    r0 = torch.sqrt(-2.0 * torch.log(1.0 - u(1, 2)))
    r1 = torch.sqrt(-2.0 * torch.log(1.0 - u(2, 2)))
    a, b = 2 * math.pi * u(2, 0), 2 * math.pi * u(3, 0)
    return (u(0, 0), u(0, 2), u(1, 0)), (r0 * torch.cos(a), r0 * torch.sin(a), r1 * torch.cos(b))


def stored(fp64, x, top=False):
    """A drawn number as the numeric form keeps it."""
    if fp64:
        return x
    x = x.to(torch.float32)
    return (x.clamp(max=0.99999994) if top else x).to(F8)


def born(c, fp64, sp, event, idx, cell, drift, flat):
    """Particles `idx` in the cells `cell` (array indices per axis); in 2D
    (flat) without y and with vy = 0."""
    u, n = drawn(c.seed, sp, event, idx)
    axes = (0, 2) if flat else (0, 1, 2)
    x = [(k.to(F8) + stored(fp64, u[0 if (flat and a == 0) else a], True)) * c.dx
         for k, a in zip(cell, axes)]
    mean = (0.0, 0.0, drift) if flat else (c.vdrift[0], c.vdrift[1], drift)
    v = []
    for a in range(3):
        if flat and a == 1:
            v.append(torch.zeros_like(n[0]))
            continue
        full = c.vth[sp] * n[a] + mean[a]
        # the rounding of the kept velocity does not depend on the drift
        v.append(full + (stored(fp64, full) - full).detach() if torch.is_tensor(full) else full)
    return x + v


def join(a, b):
    return [torch.cat((p, q)) for p, q in zip(a, b)]


def only(p, keep):
    return [q[keep] for q in p]


def lattice(x, dx, half):
    """Lower node and the two weights along one axis (truncating, as C does)."""
    h = 0.5 if half else 0.0
    k = torch.trunc(x.detach() / dx - h)
    return k.to(torch.int64), (k + 1 + h) * dx - x, x - (k + h) * dx


def stencil(shape, x, dx, halves):
    """Node indices and weights of one staggered component."""
    idx, wgt = None, None
    for a, (xa, h) in enumerate(zip(x, halves)):
        k, lo, hi = lattice(xa, dx, h)
        if idx is None:
            idx, wgt = [k, k + 1], [lo, hi]
        else:
            idx = [i * shape[a] + j for i in idx for j in (k, k + 1)]
            wgt = [v * q for v in wgt for q in (lo, hi)]
    return idx, [w / dx ** len(x) for w in wgt]


def gathered(F, x, dx, halves):
    idx, wgt = stencil(F.shape, x, dx, halves)
    f = F.reshape(-1)
    return sum(f[i] * w for i, w in zip(idx, wgt))


def deposited(acc, shape, x, dx, halves, q):
    idx, wgt = stencil(shape, x, dx, halves)
    for i, w in zip(idx, wgt):
        acc = acc.index_add(0, i, q * w) if acc.requires_grad or w.requires_grad \
            else acc.index_add_(0, i, q * w)
    return acc


def boris(c, f, v, mass, drift, relativistic):
    T = 0.5 * c.q * c.dt / mass
    e = [f[0] + drift * c.imf[1], f[1] - drift * c.imf[0], f[2]]
    b = f[3:]
    if relativistic:
        g = c.c / torch.sqrt(c.c ** 2 - v[0] ** 2 - v[1] ** 2 - v[2] ** 2)
        v = [g * a for a in v]
        g2 = c.c / torch.sqrt(c.c ** 2 + v[0] ** 2 + v[1] ** 2 + v[2] ** 2)
        b = [g2 * a for a in b]
    S = 2.0 * T / (1.0 + T * T * (b[0] ** 2 + b[1] ** 2 + b[2] ** 2))
    u = [a + p * T for a, p in zip(v, e)]
    o = [u[i] + T * (u[(i + 1) % 3] * b[(i + 2) % 3] - u[(i + 2) % 3] * b[(i + 1) % 3])
         for i in range(3)]
    u = [u[i] + S * (o[(i + 1) % 3] * b[(i + 2) % 3] - o[(i + 2) % 3] * b[(i + 1) % 3])
         + e[i] * T for i in range(3)]
    if relativistic:
        g = c.c / torch.sqrt(c.c ** 2 + u[0] ** 2 + u[1] ** 2 + u[2] ** 2)
        u = [g * a for a in u]
    return u


def depth(n, size, layer):
    """Absorber depth on the lattice of half cells, 32 cells at full width."""
    i = torch.arange(2 * size, dtype=F8, device=DEV) - 4
    if layer <= 0:
        return torch.zeros_like(i)
    d = torch.where(i <= 2 * layer, (2 * layer - i) / 4,
                    torch.where(i >= 2 * n - 2 * layer, (i - (2 * n - 2 * layer)) / 4, 0 * i))
    return d * (32.0 / layer)


def conductivity(c, n, layers):
    """sigma on the lattice of half cells as a function of the axes' parity."""
    d = [depth(a, a + 4, w) for a, w in zip(n, layers)]

    def at(parity):
        p4 = p12 = 0
        for a, q in enumerate(parity):
            s = [1] * len(n)
            s[a] = -1
            p4 = p4 + (d[a][q::2] ** 4).reshape(s)
            p12 = p12 + (d[a][q::2] ** 12).reshape(s)
        return c.sigma_amp * (0.1 * torch.sqrt(p4) + 0.01 * torch.sqrt(p12))
    return at


def shifted(F, axis, by):
    """The interior of F moved by `by` nodes along `axis`."""
    s = [slice(2, n - 2) for n in F.shape]
    if axis is not None:
        s[axis] = slice(2 + by, F.shape[axis] - 2 + by)
    return F[tuple(s)]


def d_low(F, axis):  # (2,4) difference between the nodes 0 and -1
    return (27 * (shifted(F, axis, 0) - shifted(F, axis, -1))
            - (shifted(F, axis, 1) - shifted(F, axis, -2))) / 24


def d_high(F, axis):  # between the nodes 1 and 0
    return (27 * (shifted(F, axis, 1) - shifted(F, axis, 0))
            - (shifted(F, axis, 2) - shifted(F, axis, -1))) / 24


def inner(F, new):
    F = F.clone()
    F[tuple(slice(2, n - 2) for n in F.shape)] = new
    return F


def periodic(F, axes):
    F = F.clone()
    for a in range(axes):
        n = F.shape[a] - 4
        for dst, src in ((0, n), (1, n + 1), (n + 2, 2), (n + 3, 3)):
            F.select(a, dst).copy_(F.select(a, src).clone())
    return F


class Exact3:
    """The 3D step; halves: x, y, z staggering of E (and J), B and n."""
    HE = ((0, 1, 1), (1, 0, 1), (1, 1, 0))
    HB = ((1, 0, 0), (0, 1, 0), (0, 0, 1))
    HN = (1, 1, 1)

    def __init__(self, case, seed, moment=None, drift=None):
        c = self.c = config(case, seed)
        self.case = case
        self.fp64 = case["precision"] == "fp64"
        self.n = (c.nx, c.ny, c.nz)
        self.shape = tuple(a + 4 for a in self.n)
        self.drift = c.vdrift[2] if drift is None else drift
        if moment is None:
            a = c.dipole_alpha
            moment = (0.0, c.dipole_m * math.sin(a), c.dipole_m * math.cos(a))
        self.b0 = self.dipole(moment)
        self.sigma = conductivity(c, self.n, c.absorb)
        self.event = 0

    def dipole(self, moment):
        c, out = self.c, []
        grid = torch.meshgrid(*(torch.arange(s, dtype=F8, device=DEV) - s // 2
                                for s in self.shape), indexing="ij")
        near = sum(g * g for g in grid) < c.dipole_rmax ** 2
        for a in range(3):
            r = [(g + (0.5 if a == b else 0.0)) * c.dx for b, g in enumerate(grid)]
            d = torch.sqrt(sum(q * q for q in r))
            if c.dipole_soft > 0:
                s = torch.where(d < c.dipole_soft * c.dx, c.dipole_soft * c.dx / d, 1.0 + 0 * d)
                r = [q * s for q in r]
                d = torch.sqrt(sum(q * q for q in r))
            mr = sum(m * q for m, q in zip(moment, r))
            b = c.mu0 * (3 * r[a] * mr - moment[a] * d * d) / (4 * math.pi * d ** 5)
            out.append(torch.where(near, b, 0 * b) + c.imf[a])
        return out

    def load(self):
        c, parts = self.c, []
        n = c.nx * c.ny * c.nz * c.ppc
        for sp in (0, 1):
            i = torch.arange(n, device=DEV)
            cell = i // c.ppc
            at = (cell // (c.nz * c.ny) + 2, cell // c.nz % c.ny + 2, cell % c.nz + 2)
            parts.append(born(c, self.fp64, sp, 0, i, at, self.drift, False))
        return parts

    def inflow(self, parts):
        c, out = self.c, []
        self.event += 1
        face = c.nx * c.ny * 2 * c.ppc
        i = torch.arange(face * (2 if c.refill_far else 1), device=DEV)
        r = i % face
        m = r // c.ppc % 2
        at = (r // (2 * c.ppc * c.ny) + 2, r // (2 * c.ppc) % c.ny + 2,
              torch.where(i < face, m + 2, m + c.nz))
        for sp, p in enumerate(parts):
            z = p[2].detach()
            p = only(p, ~((z < 4 * c.dx) | (z > c.nz * c.dx)))
            out.append(join(p, born(c, self.fp64, sp, self.event, i, at, self.drift, False)))
        return out

    def half_b(self, E, B):
        c, t = self.c, 0.25 * self.c.dt / self.c.eps0
        curl = (d_low(E[2], 1) - d_low(E[1], 2), d_low(E[0], 2) - d_low(E[2], 0),
                d_low(E[1], 0) - d_low(E[0], 1))
        out = []
        for a in range(3):
            s = shifted(self.sigma(self.HB[a]), None, 0) * t
            b0 = shifted(self.b0[a], None, 0)
            out.append(periodic(inner(B[a], b0 + (1 - s) / (1 + s) * (shifted(B[a], None, 0) - b0)
                                      - 0.5 * c.dt / (1 + s) * curl[a] / c.dx), 2))
        return out

    def full_e(self, E, B, J):
        c, t = self.c, self.c.c ** 2 * self.c.dt
        b = [B[a] - self.b0[a] for a in range(3)]
        curl = (d_high(b[2], 1) - d_high(b[1], 2), d_high(b[0], 2) - d_high(b[2], 0),
                d_high(b[1], 0) - d_high(b[0], 1))
        out = []
        for a in range(3):
            s = 0.5 * c.mu0 * t * shifted(self.sigma(self.HE[a]), None, 0)
            j = shifted(J[a] - J[3 + a], None, 0)
            out.append(periodic(inner(E[a], (1 - s) / (1 + s) * shifted(E[a], None, 0)
                                      + t / (1 + s) * (curl[a] / c.dx - c.mu0 * j)), 2))
        return out

    def poisson(self, E, n):
        c, A = self.c, self.c.phi_margin
        div = sum(d_high(E[a], a) for a in range(3)) / c.dx
        rho = c.q * shifted(n[0] - n[1], None, 0) / c.eps0 - div
        at = torch.meshgrid(*(torch.arange(a, device=DEV) for a in self.n), indexing="ij")
        ok = (at[2] >= A) & (at[2] < self.n[2] - A)
        for a in (0, 1):
            ok = ok & (at[a] > A) & (at[a] < self.n[a] - A)
        phi = torch.zeros(self.shape, dtype=F8, device=DEV)
        phi = periodic(inner(phi, dirichlet(torch.where(ok, rho, 0 * rho), c.dx)), 2)
        return [periodic(inner(E[a], shifted(E[a], None, 0) + d_low(phi, a) / c.dx), 2)
                for a in range(3)]

    def fields_at(self, E, B, x):
        return [gathered(F, x, self.c.dx, h) for F, h in
                zip(list(E) + list(B), self.HE + self.HB)]

    def push(self, E, B, p, sp, J, N):
        """One species, a chunk of particles: moved, deposited, those that left
        the box dropped."""
        c = self.c
        x, v = p[:3], p[3:]
        free = torch.zeros_like(x[0], dtype=torch.bool)
        for a in range(3):
            free |= (x[a].detach() < c.ballistic_lo[a]) | (x[a].detach() > c.ballistic_hi[a])
        mass = c.mass[0] if sp == 0 else -c.mass[1]
        u = boris(c, self.fields_at(E, B, x), v, mass, self.drift, True)
        v = [torch.where(free, a, b) for a, b in zip(v, u)]
        x = [a + b * c.dt * 0.5 for a, b in zip(x, v)]
        for a in range(3):
            J[3 * sp + a] = deposited(J[3 * sp + a], self.shape, x, c.dx, self.HE[a],
                                      c.q * c.weight[sp] * v[a])
        x = [a + b * c.dt * 0.5 for a, b in zip(x, v)]
        N[sp] = deposited(N[sp], self.shape, x, c.dx, self.HN, c.weight[sp] + 0 * x[0])
        keep = (x[2].detach() < (c.nz + 2) * c.dx) & (x[2].detach() >= 2 * c.dx)
        for a in (0, 1):
            L = self.n[a]
            x[a] = x[a] - L * c.dx * (x[a].detach() >= (L + 2) * c.dx) \
                + L * c.dx * (x[a].detach() < 2 * c.dx)
        return only(x + v, keep)

    def fold(self, F):
        F = F.reshape(self.shape).clone()
        for a in (0, 1):
            n = self.n[a]
            for dst, src in ((2, n + 2), (3, n + 3), (n, 0), (n + 1, 1)):
                F.select(a, dst).add_(F.select(a, src).clone())
        return F

    def step(self, E, B, parts):
        zero = torch.zeros(math.prod(self.shape), dtype=F8, device=DEV)
        J, N = [zero.clone() for _ in range(6)], [zero.clone() for _ in range(2)]
        B = self.half_b(E, B)
        out = []
        for sp, p in enumerate(parts):
            got = [self.push(E, B, [q[i:i + CHUNK] for q in p], sp, J, N)
                   for i in range(0, p[0].numel(), CHUNK)]
            out.append([torch.cat(q) for q in zip(*got)] if got else p)
        B = self.half_b(E, B)
        J, N = [self.fold(F) for F in J], [self.fold(F) for F in N]
        return self.full_e(E, B, J), B, out, J, N

    def force(self, E, B, parts):
        """The Lorentz force on the particles of the central box."""
        c, F = self.c, torch.zeros(27, dtype=F8, device=DEV)
        for sp, p in enumerate(parts):
            box = torch.ones_like(p[0], dtype=torch.bool)
            for a in range(3):
                box &= (p[a] > 0.2 * self.n[a] * c.dx) & (p[a] < 0.8 * self.n[a] * c.dx)
            p = only(p, box)
            f = torch.zeros(6, dtype=F8, device=DEV)
            for i in range(0, p[0].numel(), CHUNK):
                q = [a[i:i + CHUNK] for a in p]
                e = self.fields_at(E, B, q[:3])
                v, b = q[3:], e[3:]
                f += torch.stack([a.sum() for a in e[:3]] + [
                    (v[(a + 1) % 3] * b[(a + 2) % 3] - v[(a + 2) % 3] * b[(a + 1) % 3]).sum()
                    for a in range(3)])
            f = f * (c.q if sp == 0 else -c.q) * c.weight[sp] * c.dx ** 3
            F[3 + 6 * sp:9 + 6 * sp] += f
            F[0:3] += f[:3] + f[3:]
        return F

    def run(self, steps):
        c = self.c
        E = [torch.zeros(self.shape, dtype=F8, device=DEV) for _ in range(3)]
        B = [b.clone() for b in self.b0]
        parts = self.inflow(self.load())
        F = torch.zeros(27, dtype=F8, device=DEV)
        for s in range(steps):
            if s > 0 and s % c.inflow_every == 0:
                parts = self.inflow(parts)
            E, B, parts, J, N = self.step(E, B, parts)
            if c.poisson_every > 0 and s % c.poisson_every == 0:
                E = self.poisson(E, N)
            if self.case["thrust"]:
                F += self.force(E, B, parts)
        out = dict(zip(PLANES, [q.cpu().numpy() for q in E + B + J + N]))
        out["particles"] = np.array([float(p[0].numel()) for p in parts])
        if self.case["thrust"]:
            out["thrust"] = F.cpu().numpy()
        return out

    def flux(self, E, B):
        """Maxwell-stress z flux through the sphere around the dipole."""
        c, nq, R = self.c, self.case["points"], self.case["radius"] * self.c.dx
        q = torch.arange(nq, dtype=F8, device=DEV)
        z = 1.0 - (2.0 * q + 1.0) / nq
        r = torch.sqrt(1.0 - z * z)
        t = q * math.pi * (3.0 - math.sqrt(5.0))
        n = [r * torch.cos(t), r * torch.sin(t), z]
        x = [(s // 2) * c.dx + R * a for s, a in zip(self.shape, n)]
        f = self.fields_at(E, B, x)
        e, b = f[:3], f[3:]
        en, bn = (sum(p * a for p, a in zip(g, n)) for g in (e, b))
        e2, b2 = (sum(p * p for p in g) for g in (e, b))
        s = c.eps0 * (e[2] * en - 0.5 * z * e2) + (b[2] * bn - 0.5 * z * b2) / c.mu0
        return (s * 4 * math.pi * R * R / nq).sum()


def dirichlet(rho, dx):
    """Solve the 3- (per axis) point Laplacian with zeros at index 0 and N."""
    sym, S = 0, []
    for a, n in enumerate(rho.shape):
        k = torch.arange(n, dtype=F8, device=DEV)
        jk = torch.outer(torch.arange(n, device=DEV), torch.arange(n, device=DEV)) % (2 * n)
        S.append(torch.sin(math.pi * jk.to(F8) / n))
        shape = [1] * rho.dim()
        shape[a] = n
        sym = sym - ((torch.sin(math.pi * k / n / 2) / (dx / 2)) ** 2).reshape(shape)
    f = rho
    for a in range(rho.dim()):
        f = torch.movedim(torch.tensordot(f, S[a], dims=([a], [0])), -1, a)
    f = torch.where(sym == 0, 0 * f, f / torch.where(sym == 0, 1.0 + 0 * sym, sym))
    for a, n in enumerate(rho.shape):
        f = torch.movedim(torch.tensordot(f, S[a], dims=([a], [0])), -1, a) * (2.0 / n)
    return f


class Exact2:
    """The 2D3V step: x (k) periodic, z (m) the flow axis."""
    HE = ((0, 1), (1, 1), (1, 0))
    HB = ((1, 0), (0, 0), (0, 1))
    HN = (1, 1)

    def __init__(self, case, seed):
        c = self.c = config(case, seed)
        self.case = case
        self.fp64 = case["precision"] == "fp64"
        self.n = (c.nx, c.nz)
        self.shape = (c.nx + 4, c.nz + 4)
        self.b0 = [torch.full(self.shape, c.imf[a], dtype=F8, device=DEV) for a in range(3)]
        self.sigma = conductivity(c, self.n, c.absorb)
        self.event = 0

    def load(self):
        c, parts = self.c, []
        tx, tz = c.tile[0] or c.nx, c.tile[1] or c.nz
        ntz = c.nz // tz
        i = torch.arange(c.nx * c.nz * c.ppc, device=DEV)
        key = i // c.ppc
        tile, at = key // (tx * tz), key % (tx * tz)
        cell = (tile // ntz * tx + at // tz + 2, tile % ntz * tz + at % tz + 2)
        for sp in (0, 1):
            parts.append(self.placed(born(c, self.fp64, sp, 0, i, cell, c.vdrift, True)))
        return parts

    def placed(self, p):
        return p

    def inflow(self, parts):
        c, out = self.c, []
        self.event += 1
        face = c.nx * c.ppc
        i = torch.arange(2 * face, device=DEV)
        cell = (i % face // c.ppc + 2, torch.where(i < face, 2 + 0 * i, c.nz + 1 + 0 * i))
        for sp, p in enumerate(parts):
            p = only(p, ~((p[1] < 3 * c.dx) | (p[1] > (c.nz + 1) * c.dx)))
            out.append(join(p, born(c, self.fp64, sp, self.event, i, cell, c.vdrift, True)))
        return out

    def half_b(self, E, B):
        c = self.c
        # By uses sigma at (2k, 2m), Bx and Bz at their own nodes
        t = 0.25 * c.dt / c.eps0
        curl = (-d_low(E[1], 1), d_low(E[0], 1) - d_low(E[2], 0), d_low(E[1], 0))
        out = []
        for a in range(3):
            s = shifted(self.sigma(self.HB[a]), None, 0) * t
            b0 = shifted(self.b0[a], None, 0)
            out.append(periodic(inner(B[a], b0 + (1 - s) / (1 + s) * (shifted(B[a], None, 0) - b0)
                                      - 0.5 * c.dt / (1 + s) * curl[a] / c.dx), 1))
        return out

    def full_e(self, E, B, J):
        c, t = self.c, self.c.c ** 2 * self.c.dt
        b = [B[a] - self.b0[a] for a in range(3)]
        curl = (-d_high(b[1], 1), d_high(b[0], 1) - d_high(b[2], 0), d_high(b[1], 0))
        out = []
        for a in range(3):
            s = 0.5 * c.mu0 * t * shifted(self.sigma(self.HE[a]), None, 0)
            j = shifted(J[a] - J[3 + a], None, 0)
            out.append(periodic(inner(E[a], (1 - s) / (1 + s) * shifted(E[a], None, 0)
                                      + t / (1 + s) * (curl[a] / c.dx - c.mu0 * j)), 1))
        return out

    def poisson(self, E, n):
        c = self.c
        rho = c.q * (n[0] - n[1]) / c.eps0
        rho = shifted(rho, None, 0) - (shifted(E[0], 0, 1) - shifted(E[0], 0, 0)
                                       + shifted(E[2], 1, 1) - shifted(E[2], 1, 0)) / c.dx
        at = [torch.arange(a, device=DEV) + 2 for a in self.n]
        ok = ((at[0] >= c.phi_lo[0]) & (at[0] < c.phi_hi[0]))[:, None] \
            & ((at[1] >= c.phi_lo[1]) & (at[1] < c.phi_hi[1]))[None, :]
        phi = dirichlet(torch.where(ok, rho, 0 * rho), c.dx)
        left = torch.cat((0 * phi[:, :1], phi[:, :-1]), 1)
        ex = shifted(E[0], None, 0) + (phi - torch.roll(phi, 1, 0)) / c.dx
        ez = shifted(E[2], None, 0) + (phi - left) / c.dx
        return [periodic(inner(E[0], ex), 1), E[1], periodic(inner(E[2], ez), 1)]

    def gate(self, x):
        c = self.c
        return (x[0] < (c.nx + 3) * c.dx) & (x[0] >= c.dx) & (x[1] < (c.nz + 2) * c.dx) \
            & (x[1] >= 2 * c.dx)

    def deposit_n(self, x, sp, N):
        g = self.gate(x)
        x = only(x, g)
        N[sp] = deposited(N[sp], self.shape, x, self.c.dx, self.HN, self.c.weight[sp] + 0 * x[0])

    def push(self, E, B, p, sp, J, N):
        c = self.c
        x, v = p[:2], p[2:]
        free = torch.zeros_like(x[0], dtype=torch.bool)
        for a in range(2):
            free |= (x[a] < c.ballistic_lo[a]) | (x[a] > c.ballistic_hi[a])
        f = [gathered(F, x, c.dx, h) for F, h in zip(list(E) + list(B), self.HE + self.HB)]
        mass = c.mass[0] if sp == 0 else -c.mass[1]
        u = boris(c, f, v, mass, c.vdrift, False)
        v = [torch.where(free, a, b) for a, b in zip(v, u)]
        x = [x[0] + v[0] * c.dt * 0.5, x[1] + v[2] * c.dt * 0.5]
        g = self.gate(x)
        xg, vg = only(x, g), only(v, g)
        for a in range(3):
            J[3 * sp + a] = deposited(J[3 * sp + a], self.shape, xg, c.dx, self.HE[a],
                                      c.q * c.weight[sp] * vg[a])
        x = [x[0] + v[0] * c.dt * 0.5, x[1] + v[2] * c.dt * 0.5]
        self.deposit_n(x, sp, N)
        box = c.nx * c.dx
        inside = (x[1] < (c.nz + 2) * c.dx) & (x[1] >= 2 * c.dx)
        up = inside & (x[0] < (c.nx + 3) * c.dx) & (x[0] >= (c.nx + 2) * c.dx)
        down = inside & ~up & (x[0] > c.dx) & (x[0] < 2 * c.dx)
        x[0] = x[0] - box * up + box * down
        keep = inside & (x[0] >= 2 * c.dx) & (x[0] < (c.nx + 2) * c.dx)
        return only(x + v, keep)

    def fold(self, F):
        F = F.reshape(self.shape)
        n = self.c.nx
        F[2] += F[n + 2]
        F[n + 1] += F[1]
        return F

    def run(self, steps):
        c = self.c
        size = math.prod(self.shape)

        def zeros(k):
            return [torch.zeros(size, dtype=F8, device=DEV) for _ in range(k)]

        E = [f.reshape(self.shape) for f in zeros(3)]
        B = [b.clone() for b in self.b0]
        parts = self.load()
        N = zeros(2)
        for sp, p in enumerate(parts):
            for i in range(0, p[0].numel(), CHUNK):
                self.deposit_n([q[i:i + CHUNK] for q in p[:2]], sp, N)
        N = [periodic(self.fold(F), 1) for F in N]
        if c.poisson_every > 0:
            E = self.poisson(E, N)
        for s in range(steps):
            if c.inflow_every > 0 and s > 0 and s % c.inflow_every == 0:
                parts = self.inflow(parts)
            B = self.half_b(E, B)
            J, N, out = zeros(6), zeros(2), []
            for sp, p in enumerate(parts):
                got = [self.push(E, B, [q[i:i + CHUNK] for q in p], sp, J, N)
                       for i in range(0, p[0].numel(), CHUNK)]
                out.append([torch.cat(q) for q in zip(*got)])
            parts = out
            J, N = [self.fold(F) for F in J], [self.fold(F) for F in N]
            if c.ext_k >= 0:  # the line currents, assigned after the fold
                I = c.ext_current / c.dx ** 2
                if s < c.ext_ramp:
                    I *= (1.0 + math.cos(math.pi * s / c.ext_ramp - math.pi)) / 2
                J[1][c.ext_k, c.ext_m[0]], J[1][c.ext_k, c.ext_m[1]] = -I, I
            B = self.half_b(E, B)
            E = self.full_e(E, B, J)
            # the exchange copies whole cells: J and n guards with them
            J, N = [periodic(F, 1) for F in J], [periodic(F, 1) for F in N]
            if c.poisson_every > 0 and s % c.poisson_every == 0:
                E = self.poisson(E, N)
        out = dict(zip(PLANES, [q.cpu().numpy() for q in E + B + J + N]))
        out["particles"] = np.array([float(p[0].numel()) for p in parts])
        return out


def exact_gradient(case, seed):
    """Loss and gradient of the adjoint's window by reverse-mode autograd, each
    step's graph rebuilt from its start when it is needed."""
    from torch.utils.checkpoint import checkpoint
    c = config(case, seed)
    p = torch.tensor(parameters(case, seed, c), dtype=F8, device=DEV, requires_grad=True)
    S = Exact3(case, seed, moment=(p[0], p[1], p[2]), drift=p[3])
    E = [torch.zeros(S.shape, dtype=F8, device=DEV) for _ in range(3)]
    B = [b.clone() for b in S.b0]
    parts = S.inflow(S.load())
    loss = 0.0

    def one(*a):
        S.b0, S.drift = list(a[:3]), a[3]
        e, b, q, _, _ = S.step(a[4:7], a[7:10], (list(a[10:16]), list(a[16:22])))
        return (*e, *b, *q[0], *q[1])

    b0, drift = S.b0, S.drift
    for s in range(case["steps"]):
        if s > 0 and s % c.inflow_every == 0:
            S.drift = drift
            parts = S.inflow(parts)
        out = checkpoint(one, *b0, drift, *E, *B, *parts[0], *parts[1], use_reentrant=False)
        E, B, parts = out[0:3], out[3:6], [list(out[6:12]), list(out[12:18])]
        loss = loss + S.flux(E, B) / case["steps"]
    loss.backward()
    return {"loss": float(loss.detach()), "grad": p.grad.cpu().numpy()}


def exact(case, seed):
    n = 2 * case["nx"] * case.get("ny", 1) * case["nz"] * case["ppc"] * case["steps"]
    if case["kind"] == "adjoint":
        return exact_gradient(case, seed) if n <= 3e7 else None
    if n > 8e8:
        return None
    with torch.no_grad():
        return (Exact2 if case["kind"] == "step2d" else Exact3)(case, seed).run(case["steps"])
