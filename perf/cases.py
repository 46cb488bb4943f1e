"""The work that users of this solver have it do, as cases that can be timed.

Three ways in are covered, each through the package's public entry points:

  whole calls   `Solver(case).run()` on the small grids of the command line's
                users (every launch counts), and beams queued on a `Server`;
  depth march   `Solver.advance` on a beam resident in HBM, from the command
                line's default grid to the paper's 81 x 81 nodes, in FP32 and
                in FP64, in one material, in layers and under a material map;
  operators     the seam of `bfpn_gpu_amd.ops` (energy, transport, angle,
                secondary source, dose), as a host program with its own depth
                loop calls them.

The operators take torch tensors as their device arrays, work in place and
share the default stream, so a pass never waits for the device unless the
operator itself returns a host value.
"""
from __future__ import annotations

import ctypes
import functools
import math

import numpy as np
import torch

import bfpn_gpu_amd as bg
from bfpn_gpu_amd.abi import MATERIAL_DENSITY, Case

LG = 259.0  # the energy grid of every configuration here: [1, 260] MeV


def listed():
    return [
        # The reference's own timing case: water, 100 MeV, 9 x 9 nodes, 7 x 7
        # directions, 400 depth steps.  A whole solve, tables and all, as a
        # parameter study runs it: launch latency is what counts.
        dict(name="solve small", kind="solve", Ny=8, Nz=8, Nmu=7, Nom=7, Ng=500, Nx=2000,
             energy=100.0, material="water", precision="fp32", straggling=False, steps=400),
        # The command line's default grid: 11 x 11 nodes, 11 x 11 directions.
        dict(name="march default", kind="march", Ny=10, Nz=10, Nmu=11, Nom=11, Ng=500, Nx=4000,
             energy=230.0, material="water", precision="fp32", straggling=False, medium="one",
             steps=40),
        # One clinical beam: 21 x 21 nodes, 20 x 20 directions.
        dict(name="march beam", kind="march", Ny=20, Nz=20, Nmu=20, Nom=20, Ng=500, Nx=2000,
             energy=230.0, material="water", precision="fp32", straggling=True, medium="one",
             steps=10),
        # The paper's grid, the largest run: 1.3e9 cells, 52 GB resident.
        dict(name="march paper", kind="march", Ny=80, Nz=80, Nmu=20, Nom=20, Ng=500, Nx=4000,
             energy=230.0, material="water", precision="fp32", straggling=True, medium="one",
             steps=4),
        # The FP64 run that FP32 results are validated against.
        dict(name="march fp64", kind="march", Ny=20, Nz=20, Nmu=20, Nom=20, Ng=500, Nx=2000,
             energy=230.0, material="water", precision="fp64", straggling=True, medium="one",
             steps=2),
        # Beamlets of a treatment plan, queued on the batching server.
        dict(name="serve beamlets", kind="serve", Ny=20, Nz=20, Nmu=20, Nom=20, Ng=300, Nx=2000,
             energy=150.0, material="water", precision="fp32", straggling=True, beams=4, steps=32),
        # Operators: the secondary's energy half step on a 41 x 41 beamlet grid.
        dict(name="energy 41x41", kind="energy", Ny=40, Nz=40, Nmu=20, Nom=20, Ng=300,
             energy=150.0, material="water", precision="fp32", straggling=True, source=True),
        # Transport on the 13 x 13 grid of the reference's accuracy runs: 81
        # directions, a ragged last direction block; psi^2 keeps its sign.
        dict(name="transport 13x13", kind="transport", Ny=12, Nz=12, Nmu=9, Nom=9, Ng=500,
             energy=230.0, material="water", precision="fp32", clip=False),
        # Angular diffusion with the default 11 x 11 directions, an odd row length.
        dict(name="angle 11x11", kind="angle", Ny=20, Nz=20, Nmu=11, Nom=11, Ng=500,
             energy=230.0, material="water", precision="fp32"),
        # The secondary source of one 20 x 20 direction beam.
        dict(name="source 21x21", kind="source", Ny=20, Nz=20, Nmu=20, Nom=20, Ng=300,
             energy=150.0, material="water", precision="fp32"),
        # Transport in FP64 at a beam's size.
        dict(name="transport fp64", kind="transport", Ny=20, Nz=20, Nmu=20, Nom=20, Ng=300,
             energy=150.0, material="water", precision="fp64", clip=True),
        # The integrated dose of all four state arrays, returned to the host.
        dict(name="dose 21x21", kind="dose", Ny=20, Nz=20, Nmu=11, Nom=11, Ng=500,
             energy=230.0, material="water", precision="fp32"),
    ]


KINDS = ["march"] * 4 + ["solve", "serve", "energy", "transport", "angle", "source", "dose"]


def draw(rng):
    kind = rng.choice(KINDS)
    precision = rng.choice(["fp32", "fp32", "fp32", "fp64"])
    c = dict(kind=kind, Ng=rng.randint(200, 500), Nx=rng.choice([1000, 2000, 4000]),
             energy=round(rng.uniform(70.0, 230.0), 2), material=rng.choice(["water", "bone"]),
             precision=precision, straggling=rng.random() < 0.6)

    def size(lo, hi):  # spread over the logarithm
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    if kind == "solve":
        c.update(Ny=size(6, 14), Nz=size(6, 14), Nmu=rng.randint(4, 9), Nom=rng.randint(4, 9),
                 steps=rng.randint(100, 300), precision="fp32")
        return c
    same = rng.random() < 0.6  # most grids are square, some are not
    c.update(Ny=size(8, 80))
    c.update(Nz=c["Ny"] if same else size(8, 80))
    c.update(Nmu=rng.randint(5, 20))
    c.update(Nom=c["Nmu"] if same else rng.randint(5, 20))
    cap = dict(march=3e8, serve=6e7, energy=4e8, transport=4e8, angle=4e8, source=2e8, dose=2e8)[kind]
    cap *= 0.25 if precision == "fp64" else 1.0
    while cells(c) > cap:
        c.update(Ny=max(8, int(c["Ny"] * 0.8)), Nz=max(8, int(c["Nz"] * 0.8)))
        if c["Ny"] == 8 and c["Nz"] == 8:
            c.update(Nmu=max(5, c["Nmu"] - 1), Nom=max(5, c["Nom"] - 1))
    if kind == "march":
        c.update(medium=rng.choice(["one", "one", "one", "layers", "map"]),
                 steps=max(1, min(40, int(4e8 * (0.25 if precision == "fp64" else 1.0) / cells(c)))))
    elif kind == "serve":
        c.update(beams=rng.randint(2, 6), precision="fp32")
        c.update(steps=max(6, min(48, int(3e9 / cells(c) / c["beams"]))))
    elif kind == "energy":
        c.update(source=rng.random() < 0.5)
    elif kind == "transport":
        c.update(clip=rng.random() < 0.5)
    return c


# ------------------------------------------------------------------ sizes ---

def nodes(c):
    return (c["Ny"] + 1) * (c["Nz"] + 1)


def directions(c):
    return c["Nmu"] * c["Nom"]


def cells(c):
    return c["Ng"] * nodes(c) * directions(c)


def elem(c):
    return 8 if c["precision"] == "fp64" else 4


def dtypes(c):
    return (torch.float64, np.float64) if elem(c) == 8 else (torch.float32, np.float32)


def active(c):
    """Cells up to the beam's energy: the state above is zero."""
    top = min(1.0, (c["energy"] + 4.0) / (1.0 + LG))
    return cells(c) * top


def work(c):
    """Bytes and operations that the path cannot do without.

    A depth step has to read and write the two coefficients of both species;
    its operations are eight transports (two stages of about 24 operations),
    four sine sandwiches, ten energy half sweeps of one lane and the two
    contractions of the source."""
    n, b, na = active(c), elem(c), directions(c)
    sandwich = 4.0 * (c["Nmu"] + c["Nom"])
    step = 8 * 48 + 4 * sandwich + 8 * 28 + 4 * 0.4 * na + 2 * 60
    kind = c["kind"]
    if kind in ("march", "solve"):
        return {"bytes": 8 * b * n * c["steps"], "flops": step * n * c["steps"]}
    if kind == "serve":
        return {"bytes": 8 * b * n * c["steps"] * c["beams"],
                "flops": step * n * c["steps"] * c["beams"]}
    n = cells(c)
    if kind == "energy":
        return {"bytes": (4 + bool(c["source"])) * b * n, "flops": 28 * n}
    if kind == "transport":
        return {"bytes": 2 * b * n, "flops": 48 * n}
    if kind == "angle":
        return {"bytes": 2 * b * n, "flops": sandwich * n}
    if kind == "source":
        return {"bytes": 3 * b * n + 8 * c["Ng"] * na * na, "flops": (4 * na + 200) * n}
    return {"bytes": 4 * b * n, "flops": 8 * n}


# ----------------------------------------------------- contexts and tables ---

def beam(c, rng):
    """The beam of one request: energy and width vary a little from one to the next."""
    flags = dict(discrete_angle_delta=1, normalize_initial_mass=1, trapezoidal_yz=1,
                 eq15_straggling=int(c["straggling"]))
    dt = 40.0 / c["Nx"]
    return Case(Nx=c["Nx"], Ny=c["Ny"], Nz=c["Nz"], Ng=c["Ng"], Nmu=c["Nmu"], Nom=c["Nom"],
                Ly=8.0, Lz=8.0, Lu=2.0, Lv=2.0, Lg=LG,
                energy=c["energy"] * float(1.0 - 0.02 * rng.random()),
                sigma_yz=float(0.3 + 0.2 * rng.random()), material=c["material"],
                data=bg.tables.material_dir(c["material"]), time=c["steps"] * dt, flags=flags)


def slabs(c, other, rng):
    """Layers of two materials whose boundaries fall inside the run."""
    dt = 40.0 / c["Nx"]
    d = [(m, MATERIAL_DENSITY[m], bg.tables.material_dir(m)) for m in (c["material"], other)]
    return [(2.5 * dt,) + d[0], ((4 + rng.integers(0, 3)) * dt,) + d[1], (1e9,) + d[0]]


def insert(c, other, rng):
    """A map: a box of the other material in the middle of the plane."""
    d = [(m, MATERIAL_DENSITY[m], bg.tables.material_dir(m)) for m in (c["material"], other)]
    m = np.zeros((c["Nz"] + 1, c["Ny"] + 1), np.uint8)
    y, z = c["Ny"] // 2, c["Nz"] // 2
    k = 1 + int(rng.integers(0, max(1, c["Ny"] // 8)))
    m[z - k:z + k + 1, y - k:y + k + 1] = 1
    return d, [1e9], m.reshape(1, -1)


@functools.lru_cache(maxsize=4)
def physics(Ng, material):
    """The per-group tables, which a host program has from its own set-up."""
    c = Case(Nx=100, Ny=1, Nz=1, Ng=Ng, Nmu=1, Nom=1, Lg=LG, material=material,
             data=bg.tables.material_dir(material))
    with bg.Solver(c, bg.FP64) as s:
        return {k: s.table(k) for k in ("S", "sigma", "T", "sig_tr", "en")}


@functools.lru_cache(maxsize=1)
def kernels(Ng, Nmu, Nom, material):
    """The source's energy and angular kernels of one grid and material."""
    c = Case(Nx=100, Ny=1, Nz=1, Ng=Ng, Nmu=Nmu, Nom=Nom, Lu=2.0, Lv=2.0, Lg=LG, material=material,
             data=bg.tables.material_dir(material))
    with bg.Solver(c, bg.FP64) as s:
        t = {k: s.table(k) for k in ("ker_e1", "ker_e2", "ker_v")}
        t.update({k: s.table(k).astype(np.int32) for k in ("ker_beg", "ker_end")})
        return t


def deltas(c):
    return dict(dt=0.02, dy=8.0 / c["Ny"], dz=8.0 / c["Nz"], dg=LG / c["Ng"],
                du=2.0 / (c["Nom"] + 1), dv=2.0 / (c["Nmu"] + 1))


def velocities(c):
    """(omega_y, omega_z) of every direction, the solver's order."""
    d = deltas(c)
    v = -1.0 + (c["Nmu"] - np.arange(c["Nmu"])) * d["dv"]
    u = -1.0 + (np.arange(c["Nom"]) + 1) * d["du"]
    return np.stack(np.broadcast_arrays(-v[:, None], -u[None, :]), axis=-1).reshape(-1)


class Held:
    """A torch tensor as the operators' device array (they read ptr and dtype)."""

    def __init__(self, t, dtype):
        self.t, self.dtype, self.ptr = t, np.dtype(dtype), ctypes.c_void_p(t.data_ptr())


def on_gpu(a):
    a = np.ascontiguousarray(a)
    return Held(torch.from_numpy(a).cuda(), a.dtype)


def field(c, gen, signed):
    """A beam's phase space [g][s][m]: a spectrum around the energy it has left
    with a tail below, a Gaussian spot, a forward cone, and 10 % of noise.
    signed: psi^2, of both signs and about a fifth as large."""
    dt, _ = dtypes(c)
    o = dict(device="cuda", dtype=torch.float32)
    E = 1.0 + (torch.arange(c["Ng"], **o) + 0.5) * (LG / c["Ng"])
    E0 = c["energy"] * 0.9
    spec = torch.exp(-0.5 * ((E - E0) / 4.0) ** 2) + 0.02 * (E < E0)
    y = torch.linspace(-4.0, 4.0, c["Ny"] + 1, **o)
    z = torch.linspace(-4.0, 4.0, c["Nz"] + 1, **o)
    spot = torch.exp(-0.5 * ((z[:, None] - 0.3) ** 2 + (y[None, :] + 0.2) ** 2)).reshape(-1)
    w = torch.from_numpy(velocities(c)).cuda().float().reshape(-1, 2)
    cone = torch.exp(-(w ** 2).sum(1) / 0.08)
    lane = (spot[:, None] * cone[None, :]).reshape(-1)
    out = torch.empty((c["Ng"], lane.numel()), device="cuda", dtype=dt)
    for g in range(0, c["Ng"], 16):
        r = torch.rand((min(16, c["Ng"] - g), lane.numel()), generator=gen, **o)
        r = 0.2 * (2.0 * r - 1.0) if signed else 1.0 + 0.2 * (r - 0.5)
        out[g:g + 16] = (spec[g:g + 16, None] * lane[None, :] * r).to(dt)
    return out.reshape(-1)


def prepare(c, seed):
    rng = np.random.default_rng(seed)
    kind = c["kind"]
    prec = bg.FP64 if elem(c) == 8 else bg.FP32
    if kind == "solve":
        return dict(c=c, beam=beam(c, rng), prec=prec)
    if kind == "march":
        other = "bone" if c["material"] == "water" else "water"
        extra = {}
        if c["medium"] == "layers":
            extra["layers"] = slabs(c, other, rng)
        elif c["medium"] == "map":
            extra["mapped"] = insert(c, other, rng)
        return dict(c=c, solver=bg.Solver(beam(c, rng), prec, **extra))
    if kind == "serve":
        server = bg.Server(max_active=8, slice_steps=32, precision=prec)
        # a running service has the tables of its grid in its cache
        first = beam(c, rng)
        server.wait(server.submit(first, first.dt))
        return dict(c=c, server=server, beams=[beam(c, rng) for _ in range(c["beams"])])
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    ty = dtypes(c)[1]
    st = dict(c=c, ws=bg.Workspace(), d=deltas(c))
    F = Held(field(c, gen, False), ty)
    if kind == "angle":
        st.update(F=F, sig_tr=physics(c["Ng"], c["material"])["sig_tr"])
        return st
    if kind == "transport":
        st.update(F=F if c["clip"] else Held(field(c, gen, True), ty), om=on_gpu(velocities(c)))
        return st
    st.update(F=F, f=Held(field(c, gen, True), ty))
    st.update({k: on_gpu(v) for k, v in physics(c["Ng"], c["material"]).items()})
    if kind == "energy":
        st["Q"] = Held(field(c, gen, False) * 1e-2, ty) if c["source"] else None
    elif kind == "dose":
        st.update(F1=Held(field(c, gen, False) * 1e-2, ty), f1=Held(field(c, gen, True) * 1e-2, ty))
    elif kind == "source":
        k = kernels(c["Ng"], c["Nmu"], c["Nom"], c["material"])
        st.update({n: on_gpu(v) for n, v in k.items()})
        st["Q"] = Held(torch.zeros_like(F.t), ty)
        bg.ops.secondary_source_prepare(st["ker_e1"], st["ker_e2"], st["ker_v"], st["ker_beg"],
                                        st["ker_end"], c["Ng"], directions(c), st["d"]["dg"], ty,
                                        st["ws"])
    return st


# -------------------------------------------------------------------- run ---

def kept(c, *arrays):
    """Histories and projections of a state carry that state's precision."""
    return [np.asarray(a, dtype=dtypes(c)[1]) for a in arrays]


def run(st):
    c = st["c"]
    kind = c["kind"]
    if kind == "solve":
        # the whole call: tables, state, march, and the files' content
        with bg.Solver(st["beam"], st["prec"]) as s:
            idd, proxy = s.run()
            return kept(c, idd, proxy, s.spot_plane(), s.energy_moments())
    if kind == "march":
        # a slice of the march, then what a program saves of it: the depth
        # dose so far and, in one material or in layers, the current state's
        # dose plane and energy moments
        s = st["solver"]
        s.advance(c["steps"])
        idd, proxy = s.history()
        if c["medium"] == "map":
            return kept(c, idd, proxy)
        return kept(c, idd, proxy, s.spot_plane(), s.energy_moments())
    if kind == "serve":
        ids = [st["server"].submit(b) for b in st["beams"]]
        return kept(c, *[st["server"].wait(i)[0] for i in ids])
    d, ws, Ng, na = st["d"], st["ws"], c["Ng"], directions(c)
    if kind == "energy":
        bg.ops.energy_half(st["F"], st["f"], st["S"], st["sigma"], st["T"], 0.5 * d["dt"], d["dg"],
                           MATERIAL_DENSITY[c["material"]], Ng, nodes(c), na, Q1=st["Q"],
                           straggling=c["straggling"], ws=ws)
        return [st["F"].t, st["f"].t]
    if kind == "transport":
        bg.ops.transport_half(st["F"], st["om"], c["Ny"], c["Nz"], Ng, na, d["dy"], d["dz"],
                              0.5 * d["dt"], not c["clip"], ws=ws)
        return st["F"].t
    if kind == "angle":
        bg.ops.angle_full(st["F"], st["sig_tr"], nodes(c), Ng, c["Nmu"], c["Nom"], d["du"], d["dv"],
                          d["dt"], MATERIAL_DENSITY[c["material"]], ws=ws)
        return st["F"].t
    if kind == "source":
        bg.ops.secondary_source(st["F"], st["f"], st["Q"], st["ker_e1"], st["ker_e2"], st["ker_v"],
                                st["ker_beg"], st["ker_end"], Ng, nodes(c), na, d["dg"], ws=ws,
                                prepared=True)
        return st["Q"].t
    return bg.ops.idd(st["F"], st["f"], st["F1"], st["f1"], st["S"], st["sigma"], st["en"], Ng,
                      c["Ny"], c["Nz"], na, d["dg"], d["du"], d["dv"], d["dy"], d["dz"],
                      MATERIAL_DENSITY[c["material"]], trapezoidal=True, ws=ws)


# ------------------------------------------------------------------ exact ---

def exact(c, seed):
    """One operator application in 64 bits.  Whole marches would take minutes
    (500 sequential groups per sweep, hundreds of sweeps)."""
    if c["kind"] in ("solve", "march", "serve"):
        return None
    st = prepare(c, seed)
    return {"energy": exact_energy, "transport": exact_transport, "angle": exact_angle,
            "source": exact_source, "dose": exact_dose}[c["kind"]](c, st)


def as64(h, c):
    return h.t.double().reshape(c["Ng"], -1)


def exact_energy(c, st):
    """Eq.15: discontinuous Galerkin in energy, Crank-Nicolson in depth, one
    sweep from the highest group to the lowest."""
    t = physics(c["Ng"], c["material"])
    h, dg, rho = 0.5 * st["d"]["dt"], st["d"]["dg"], MATERIAL_DENSITY[c["material"]]
    P, R = as64(st["F"], c), as64(st["f"], c)
    Q = as64(st["Q"], c) if c["source"] else None
    zero = torch.zeros_like(P[0])
    outP, outR = torch.empty_like(P), torch.empty_like(R)
    delta = zero
    Ng = c["Ng"]
    for g in reversed(range(Ng)):
        lo, hi = max(t["S"][g], 0.0) * rho / dg, max(t["S"][g + 1], 0.0) * rho / dg
        sig = max(t["sigma"][g], 0.0)
        T = [max(t["T"][k], 0.0) * rho / dg ** 2 if c["straggling"] and 0 <= k < Ng else 0.0
             for k in (g - 1, g, g + 1)]
        Ph, Rh = (P[g + 1], R[g + 1]) if g + 1 < Ng else (zero, zero)
        inF = 1.0 / (1.0 / h + 0.5 * lo + 0.5 * sig)
        common = ((0.5 * hi + 0.5 * T[2]) * Ph - 0.5 * hi * Rh
                  + (1.0 / h - 0.5 * sig - 0.5 * lo - T[1]) * P[g] + 0.5 * lo * R[g])
        if g > 0:
            common = common + 0.5 * T[0] * P[g - 1]
        if Q is not None:
            common = common + Q[g]
        A = 1.5 * hi * inF
        rhs = (1.5 * hi * Ph - 1.5 * hi * Rh + (1.5 * lo - 1.5 * (lo + hi)) * P[g]
               + (1.0 / h - 0.5 * sig - 1.5 * lo - 0.5 * (hi - lo)) * R[g] - A * common
               + (1.5 * hi - A * 0.5 * hi) * delta)
        coe = 1.0 / h + 0.5 * sig + 1.5 * lo + 0.5 * (hi - lo) + A * 0.5 * lo
        fn = rhs / coe
        Fn = 0.5 * lo * inF * fn + inF * common + 0.5 * hi * inF * delta
        delta = Fn - fn
        outP[g], outR[g] = Fn, fn
    return [outP.reshape(-1), outR.reshape(-1)]


def exact_transport(c, st):
    """Eq.18: MUSCL reconstruction with the superbee limiter, predictor and
    corrector, clamped stencils at the plane's edges."""
    d, h = st["d"], 0.5 * st["d"]["dt"]
    w = torch.from_numpy(velocities(c)).cuda().reshape(-1, 2)
    F = as64(st["F"], c).reshape(c["Ng"], c["Nz"] + 1, c["Ny"] + 1, -1)

    def limited(left, mid, right):
        fwd = right - mid
        th = (mid - left) / torch.where(fwd.abs() < 1e-10, torch.ones_like(fwd), fwd)
        eta = torch.maximum(torch.clamp(2.0 * th, max=1.0), torch.clamp(th, max=2.0)).clamp(min=0.0)
        return torch.where(fwd.abs() < 1e-10, torch.zeros_like(fwd), fwd * eta)

    def axis(X, dim, v):
        n = X.shape[dim]
        at = lambda k: X.index_select(dim, torch.arange(n, device="cuda").add(k).clamp(0, n - 1))  # noqa: E731
        m2, m1, p1, p2 = at(-2), at(-1), at(1), at(2)
        Sm, S, Sp = limited(m2, m1, X), limited(m1, X, p1), limited(X, p1, p2)
        pos = X + 0.5 * S - (m1 + 0.5 * Sm)
        neg = p1 - 0.5 * Sp - (X - 0.5 * S)
        return v * torch.where(v >= 0.0, pos, neg)

    def flux(X):
        return axis(X, 2, w[:, 0]) / d["dy"] + axis(X, 1, w[:, 1]) / d["dz"]

    clip = (lambda x: x.clamp(min=0.0)) if c["clip"] else (lambda x: x)
    out = torch.empty_like(F)
    for g in range(0, c["Ng"], 20):
        X = F[g:g + 20]
        L = flux(X)
        out[g:g + 20] = clip(X - 0.5 * h * (L + flux(clip(X - h * L))))
    return out.reshape(-1)


def exact_angle(c, st):
    """Eq.19: Crank-Nicolson on the zero-boundary sine basis of each plane."""
    d, rho = st["d"], MATERIAL_DENSITY[c["material"]]

    def basis(n):
        k = torch.arange(1, n + 1, device="cuda", dtype=torch.float64)
        return torch.sin(math.pi * k[:, None] * k[None, :] / (n + 1)), \
            2.0 - 2.0 * torch.cos(math.pi * k / (n + 1))

    (Su, lu), (Sv, lv) = basis(c["Nom"]), basis(c["Nmu"])
    lam = lv[:, None] / d["dv"] ** 2 + lu[None, :] / d["du"] ** 2
    F = as64(st["F"], c).reshape(c["Ng"], -1, c["Nmu"], c["Nom"])
    out = torch.empty_like(F)
    norm = 4.0 / ((c["Nom"] + 1.0) * (c["Nmu"] + 1.0))
    for g in range(c["Ng"]):
        a = 0.5 * rho * float(st["sig_tr"][g]) * lam
        ratio = (2.0 / d["dt"] - a) / (2.0 / d["dt"] + a) * norm
        hat = torch.matmul(Sv, torch.matmul(F[g], Su)) * ratio
        out[g] = torch.matmul(Sv, torch.matmul(hat, Su))
    return out.reshape(-1)


def exact_source(c, st):
    """The angular contraction of each source group, then the energy kernels."""
    Ng, na, dg = c["Ng"], directions(c), st["d"]["dg"]
    Kv = st["ker_v"].t.reshape(Ng, na, na)
    A1 = as64(st["F"], c).clamp(min=0.0).reshape(Ng, -1, na)
    A2 = as64(st["f"], c).reshape(Ng, -1, na)
    for g in range(Ng):
        A1[g] = A1[g] @ Kv[g]
        A2[g] = A2[g] @ Kv[g]
    K1, K2 = st["ker_e1"].t.reshape(Ng, Ng), st["ker_e2"].t.reshape(Ng, Ng)
    return (dg * (K1 @ A1.reshape(Ng, -1) + K2 @ A2.reshape(Ng, -1) / 3.0)).reshape(-1)


def exact_dose(c, st):
    """Eq.24 with trapezoid weights on the transverse plane."""
    t = {k: st[k].t for k in ("S", "sigma", "en")}
    d = st["d"]
    sig = t["sigma"].clamp(min=0.0)
    S, en = t["S"], t["en"]
    w1 = (0.5 * (S[1:] + S[:-1]) + 0.5 * (en[1:] + en[:-1]) * sig) * d["dg"]
    w2 = ((S[1:] - S[:-1]) + (en[1:] - en[:-1]) * sig) / 6.0 * d["dg"]
    wy = torch.ones(c["Ny"] + 1, device="cuda", dtype=torch.float64)
    wz = torch.ones(c["Nz"] + 1, device="cuda", dtype=torch.float64)
    for w in (wy, wz):
        w[0] = w[-1] = 0.5
    lane = (wz[:, None] * wy[None, :]).reshape(-1).repeat_interleave(directions(c))
    total = (w1 @ ((as64(st["F"], c) + as64(st["F1"], c)) @ lane)
             + w2 @ ((as64(st["f"], c) + as64(st["f1"], c)) @ lane))
    return float(total) * d["du"] * d["dv"] * d["dy"] * d["dz"] / MATERIAL_DENSITY[c["material"]]
