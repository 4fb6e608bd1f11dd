"""The work that programs have this library do, as cases that can be timed and compared.

listed() names the cases, draw(rng) gives more of the same ranges, prepare(case, seed) makes what
a program holds before the call (a Simulation with its fields), run(state) is one
call through the Python package, work(case) the bytes and operations it cannot do without, and
exact(case, seed) the result in 64-bit torch arithmetic where one call has a closed description.

Kinds of case:
  steps      Simulation.simulate(n): whole time steps, dt on the device (how a run spends its time)
  one        calc_max_timestep + advance(dt) + the body's drag: the reference's own step loop
  gradient   adjoint_forward + adjoint_backward: mean drag and its gradient
  operators  advdiff, pressure_rhs, poisson_solve, pressure_correction called one by one
  solve      poisson_solve on a given right-hand side
Grids are given in blocks of 32 x 32 cells.
"""
import math

import numpy as np
import torch

import cubismup_2d_amd as cup

BS = 32


def _fade_len(case):
    """The package's default boundary fade of the right-hand side; none in the cosine solver's
    box, whose walls need none."""
    return 0.0 if case.get("poisson") == "cosine" else 0.01


# the benchmark's swimmer (one body length 0.2 in a domain of 2 x 1)
SWIMMER = dict(L=0.2, T=1.0, envelope="quadratic", env_a0=0.02, env_a2=0.08, waveLength=1.0,
               profile="naca", naca_t=0.08)


def listed():
    return [
        # the headline run: one free swimmer on the periodic 4096 x 2048 grid, FP64
        dict(name="steps swimmer 4096x2048", kind="steps", body="swimmer", bpdx=128, bpdy=64,
             poisson="periodic", precision="fp64", sweeps=0, n=10),
        # the same run at FP32 with its default of one FP64 refinement sweep per solve
        dict(name="steps swimmer 4096x2048 fp32", kind="steps", body="swimmer", bpdx=128, bpdy=64,
             poisson="periodic", precision="fp32", sweeps=1, n=10),
        # the scale-up run: four swimmers and sixteen disks on 8192 x 4096
        dict(name="steps mixed 8192x4096", kind="steps", body="mixed", bpdx=256, bpdy=128,
             poisson="periodic", precision="fp64", sweeps=0, n=8),
        # the towed cylinder at the reference's own size: cache-resident, bound by launches
        dict(name="steps cylinder 512x256", kind="steps", body="cylinder", bpdx=16, bpdy=8,
             poisson="freespace", precision="fp64", sweeps=0, n=20),
        # a production towed cylinder on a grid that is no power of two (padded to 4096 x 2048)
        dict(name="steps cylinder 2016x992", kind="steps", body="cylinder", bpdx=63, bpdy=31,
             poisson="freespace", precision="fp64", sweeps=0, n=10),
        # the reference's default solver (cosine): two cylinders in tandem in a box
        dict(name="steps tandem 2048x1024 cosine", kind="steps", body="tandem", bpdx=64, bpdy=32,
             poisson="cosine", precision="fp64", sweeps=0, n=10),
        # the reference's loop, one step per call with dt and drag on the host: the smallest call
        dict(name="one cylinder 256x128", kind="one", body="cylinder", bpdx=8, bpdy=4,
             poisson="freespace", precision="fp64", sweeps=0, n=1),
        # the iterative penalization (a Poisson solve per iteration, its test on the host)
        dict(name="steps iterative 1024x512", kind="steps", body="cylinder", bpdx=32, bpdy=16,
             poisson="freespace", precision="fp64", sweeps=0, n=4, iterative=True),
        # one gradient of the mean drag over a short horizon
        dict(name="gradient 512x256", kind="gradient", bpdx=16, bpdy=8, n=20, every=10, modes=16),
        # the operators called one by one (a host program with its own pipeline)
        dict(name="operators 4096x2048", kind="operators", bpdx=128, bpdy=64, poisson="periodic"),
        # the Poisson solver by itself: the default solver at an ordinary size
        dict(name="solve cosine 1024x512", kind="solve", bpdx=32, bpdy=16, poisson="cosine"),
        # and the free-space solver on the largest ragged grid it takes (padded to 8192 x 4096)
        dict(name="solve freespace 4000x2016", kind="solve", bpdx=125, bpdy=63,
             poisson="freespace"),
    ]


def _logint(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _pow2_grid(rng, lo, hi):
    bx = 2 ** rng.randint(lo, hi)
    by = max(4, bx // rng.choice((1, 2, 2, 2, 4)))
    return bx, by


def _pow2(n):
    return 1 << (n - 1).bit_length()


def _ragged_grid(rng, lo, hi):
    bx = _logint(rng, lo, hi)
    return bx, max(4, min(64, int(bx * rng.uniform(0.4, 0.6))))


def draw(rng):
    kind = rng.choice(("steps",) * 5 + ("one", "gradient", "operators", "solve", "solve"))
    if kind == "steps":
        body = rng.choice(("swimmer", "swimmer", "mixed", "cylinder", "cylinder", "tandem"))
        c = dict(kind=kind, body=body, precision="fp64", sweeps=0)
        if body in ("swimmer", "mixed"):
            bx = 2 ** rng.randint(5, 7)  # a swimmer needs a hundred cells of length
            c.update(bpdx=bx, bpdy=bx // 2, poisson="periodic")
            if body == "swimmer" and rng.random() < 0.4:
                c.update(precision="fp32", sweeps=rng.randint(0, 2))
        elif body == "cylinder":
            bx, by = _ragged_grid(rng, 8, 100)
            c.update(bpdx=bx, bpdy=by, poisson="freespace")
            option = rng.random()
            if option < 0.25:
                c.update(precision="fp32")
            elif option < 0.4:
                c.update(iterative=True)
        else:
            bx = 2 ** rng.randint(3, 7)
            c.update(bpdx=bx, bpdy=bx // 2, poisson="cosine")
        # steps per call, within the listed 8192 x 4096 run's cell-steps (of the padded or
        # mirrored grid, once more for each refinement sweep)
        cells = c["bpdx"] * c["bpdy"] * (1 + c["sweeps"])
        if body == "cylinder":
            cells = 4 * _pow2(c["bpdx"]) * _pow2(c["bpdy"]) * (8 if c.get("iterative") else 1)
        elif body == "tandem":
            cells *= 4
        c["n"] = max(1, min(rng.randint(4, 20), 8 * 256 * 128 // cells))
        return c
    if kind == "one":
        bx, by = _ragged_grid(rng, 8, 40)
        return dict(kind=kind, body="cylinder", bpdx=bx, bpdy=by, poisson="freespace",
                    precision="fp64", sweeps=0, n=1)
    if kind == "gradient":
        bx = _logint(rng, 8, 32)
        return dict(kind=kind, bpdx=bx, bpdy=max(4, bx // 2), n=rng.randint(6, 20),
                    every=rng.choice((5, 10, 20)), modes=rng.choice((4, 8, 16)))
    if kind == "operators":
        bx, by = _pow2_grid(rng, 3, 7)
        return dict(kind=kind, bpdx=bx, bpdy=by, poisson=rng.choice(("periodic", "cosine")))
    poisson = rng.choice(("periodic", "cosine", "freespace"))
    bx, by = _ragged_grid(rng, 4, 125) if poisson == "freespace" else _pow2_grid(rng, 2, 7)
    return dict(kind=kind, bpdx=bx, bpdy=by, poisson=poisson)


# ------------------------------------------------------------------ inputs
def _noise(shape, seed, scale):
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float64) * scale


def _velocity(NX, NY, h, seed, rms):
    """Random smooth solenoidal velocity (2, NY, NX) of the given rms: white vorticity filtered
    to a few tens of eddies across the domain, through its streamfunction."""
    w = torch.fft.rfft2(_noise((NY, NX), seed, 1.0))
    kx = torch.fft.rfftfreq(NX, device="cuda", dtype=torch.float64)[None, :] * (2 * math.pi)
    ky = torch.fft.fftfreq(NY, device="cuda", dtype=torch.float64)[:, None] * (2 * math.pi)
    k2 = kx * kx + ky * ky
    k2[0, 0] = 1.0
    k0 = 2 * math.pi * 24 / NX
    psi = torch.fft.irfft2(w / k2 * torch.exp(-k2 / (k0 * k0)), s=(NY, NX))
    u = (torch.roll(psi, -1, 0) - torch.roll(psi, 1, 0)) / (2 * h)
    v = -(torch.roll(psi, -1, 1) - torch.roll(psi, 1, 1)) / (2 * h)
    vel = torch.stack([u, v])
    return vel * (rms / vel.square().mean().sqrt())


def _rhs(NX, NY, h, seed):
    """A pressure right-hand side as a step forms it: (h / 2 dt) div of a velocity that is not
    quite solenoidal, here by noise of a percent."""
    vel = _velocity(NX, NY, h, seed, 0.1) + _noise((2, NY, NX), seed + 1, 1e-3)
    return _div(vel[0], vel[1]) * (0.5 * h / (0.05 * h))


def _bodies(case, rng):
    def u(a, b):
        return float(rng.uniform(a, b))
    body = case["body"]
    if body == "swimmer":
        return [cup.carlingfish(u(0.9, 1.1), u(0.45, 0.55), phi=u(0.0, 1.0), **SWIMMER)]
    if body == "cylinder":
        return [cup.disk(u(0.045, 0.055), u(0.22, 0.3), u(0.22, 0.26), xvel=u(0.15, 0.25),
                         bFixed=True, bForced=True)]
    if body == "tandem":
        U, y = u(0.15, 0.25), u(0.22, 0.28)
        return [cup.disk(0.04, u(0.2, 0.25), y, xvel=U, bFixed=True, bForced=True),
                cup.disk(0.04, u(0.45, 0.5), y + u(-0.02, 0.02), xvel=U, bFixed=True,
                         bForced=True)]
    # mixed: swimmers in the four quarters, disks on a jittered lattice along the walls between
    shapes = [cup.carlingfish(x + u(-0.03, 0.03), y + u(-0.02, 0.02), phi=u(0.0, 1.0), **SWIMMER)
              for x in (0.55, 1.45) for y in (0.35, 0.65)]
    for k in range(16):
        x, y = 0.15 + 0.24 * (k % 8) + u(-0.02, 0.02), (0.11, 0.89)[k // 8] + u(-0.02, 0.02)
        shapes.append(cup.disk(u(0.01, 0.03), x, y, bForced=True))
    return shapes


def _simulation(case, seed):
    """A run under way: bodies placed, a seeded flow made divergence-free by one projection,
    two steps taken."""
    rng = np.random.default_rng(seed)
    wide = case["body"] in ("swimmer", "mixed")  # domain 2 x 1, free bodies in a quiet flow
    sim = cup.Simulation(case["bpdx"], case["bpdy"], extent=2.0 if wide else 1.0,
                         nu=1e-5 if wide else 2e-4, CFL=0.1, fadeLen=_fade_len(case),
                         poisson=case["poisson"], precision=case["precision"],
                         refine_sweeps=case["sweeps"],
                         iterative_penal=case.get("iterative", False), shapes=_bodies(case, rng))
    sim.reset()
    vel = _velocity(sim.NX, sim.NY, sim.scalars()["h"], seed, 1e-3 if wide else 0.01)
    sim.set_field(cup.VEL, vel.cpu().numpy())
    sim.pressure_rhs(1.0)
    sim.poisson_solve()
    sim.pressure_correction(1.0)
    sim.simulate(2)
    return sim


class _Plane:
    """A device plane of a simulation for torch (no copy); keeps the simulation alive."""

    def __init__(self, sim, ptr, shape, typestr):
        self.sim = sim
        self.__cuda_array_interface__ = dict(shape=shape, typestr=typestr, data=(ptr, False),
                                             version=2)


def _plane(state, sim, field, comp=0):
    ptr = sim.device_ptr(field, comp)
    if ptr not in state["views"]:
        f32 = sim.precision == "fp32" and field in (cup.VEL, cup.TMPV, cup.TMP)
        t = torch.as_tensor(_Plane(sim, ptr, (sim.NY, sim.NX), "<f4" if f32 else "<f8"),
                            device="cuda")
        t.simulation = sim  # the tensor is a view of the simulation's memory
        state["views"][ptr] = t
    return state["views"][ptr]


def _fields(state, sim):
    """Velocity and pressure; an FP32 program keeps its pressure in float too."""
    p = _plane(state, sim, cup.PRES)
    return dict(u=_plane(state, sim, cup.VEL, 0), v=_plane(state, sim, cup.VEL, 1),
                p=p.float() if sim.precision == "fp32" else p)


def _dt(case):
    """Time step of the operator calls: 0.05 cells per step at the flow's rms speed."""
    return 0.05 * (1.0 / (BS * max(case["bpdx"], case["bpdy"]))) / 0.1


def prepare(case, seed):
    kind = case["kind"]
    st = dict(kind=kind, case=case, views={})
    if kind in ("steps", "one"):
        st["sim"] = _simulation(case, seed)
    elif kind == "gradient":
        rng = np.random.default_rng(seed)
        d = cup.disk(float(rng.uniform(0.045, 0.055)), float(rng.uniform(0.25, 0.3)),
                     float(rng.uniform(0.23, 0.27)), xvel=0.2, bFixed=True, bForced=True)
        sim = cup.Simulation(case["bpdx"], case["bpdy"], extent=1.0, nu=2e-4, CFL=0.1,
                             fadeLen=_fade_len(case), poisson="freespace", shapes=[d])
        sim.reset()
        sim.set_surface_velocity(rng.normal(0.0, 1e-3, 4 * case["modes"]))
        st["sim"] = sim
    else:
        sim = cup.Simulation(case["bpdx"], case["bpdy"], extent=1.0, nu=1e-3, CFL=0.1,
                             fadeLen=_fade_len(case), poisson=case["poisson"])
        h = sim.scalars()["h"]
        if kind == "operators":
            sim.set_field(cup.VEL, _velocity(sim.NX, sim.NY, h, seed, 0.1).cpu().numpy())
        else:
            sim.set_field(cup.TMP, _rhs(sim.NX, sim.NY, h, seed).cpu().numpy())
        st["sim"] = sim
    return st


def run(state):
    kind, case = state["kind"], state["case"]
    sim = state["sim"]
    if kind == "steps":
        sim.simulate(case["n"])
        return _fields(state, sim)
    if kind == "one":
        dt = sim.calc_max_timestep()
        sim.advance(dt)
        return dict(_fields(state, sim), dt=dt, drag=sim.shape(0)["drag"])
    if kind == "gradient":
        J, dts = sim.adjoint_forward(case["n"], case["every"])
        return dict(J=J, dts=dts, gradient=sim.adjoint_backward(),
                    u=_plane(state, sim, cup.VEL, 0), v=_plane(state, sim, cup.VEL, 1))
    if kind == "operators":
        dt = _dt(case)
        sim.advdiff(dt)
        sim.pressure_rhs(dt)
        sim.poisson_solve()
        sim.pressure_correction(dt)
        return _fields(state, sim)
    sim.poisson_solve()
    return dict(p=_plane(state, sim, cup.PRES), rhs=_plane(state, sim, cup.TMP))


def work(case):
    """Per cell and step: velocity read, velocity and pressure written; a stencil's operations
    and those of a real transform there and back (2.5 log2 n per point and direction)."""
    kind = case["kind"]
    cells, steps = float(case["bpdx"] * case["bpdy"]) * BS * BS, case.get("n", 1)
    pad = 4.0 if case.get("poisson", "freespace") == "freespace" else 1.0
    fft = 2 * 2.5 * pad * math.log2(max(2.0, pad * cells))
    if kind == "solve":
        return {"bytes": 16.0 * cells, "flops": cells * fft}
    real = 4.0 if case.get("precision") == "fp32" else 8.0
    sweeps = case.get("sweeps", 0)
    scale = 2.0 if kind == "gradient" else 1.0  # the backward sweep is a step's work again
    return {"bytes": scale * steps * cells * (4 * real + 8.0),
            "flops": scale * steps * cells * (60.0 + fft * (1 + 2 * sweeps))}


# ------------------------------------------------------- 64-bit references
def _shift(a, dx, dy):
    """Neighbour values with zero-gradient faces."""
    p = torch.nn.functional.pad(a[None, None], (1, 1, 1, 1), mode="replicate")[0, 0]
    NY, NX = a.shape
    return p[1 + dy:1 + dy + NY, 1 + dx:1 + dx + NX]


def _div(u, v):
    return _shift(u, 1, 0) - _shift(u, -1, 0) + _shift(v, 0, 1) - _shift(v, 0, -1)


def _fade(r, case, h):
    """The right-hand side faded towards the domain faces, its sum kept (cub2rhs)."""
    NY, NX = r.shape
    L, ex, ey = _fade_len(case), NX * h, NY * h
    eps = 2.220446049250313e-16
    x = (torch.arange(NX, device="cuda", dtype=torch.float64) + 0.5) * h
    y = (torch.arange(NY, device="cuda", dtype=torch.float64) + 0.5) * h
    bx, by = torch.arange(NX, device="cuda") // BS, torch.arange(NY, device="cuda") // BS
    first_x, last_x = (bx * BS + 0.5) * h, (bx * BS + BS - 0.5) * h
    first_y, last_y = (by * BS + 0.5) * h, (by * BS + BS - 0.5) * h
    band = ((L >= ex - last_x) | (L >= first_x))[None, :] | \
           ((L >= ey - last_y) | (L >= first_y))[:, None]
    ax = torch.maximum((L - ex + x).clamp(min=0), (L - x).clamp(min=0)) / max(L, eps)
    ay = torch.maximum((L - ey + y).clamp(min=0), (L - y).clamp(min=0)) / max(L, eps)
    fa2 = torch.maximum(ax[None, :], ay[:, None]).clamp(max=1).square()
    f = torch.where(band, r * fa2, torch.zeros_like(r))
    total, pos, neg = f.sum(), f.clamp(min=0).sum(), (-f).clamp(min=0).sum()
    corr = total / pos.clamp(min=eps) if total > 0 else total / neg.clamp(min=eps)
    back = corr * (f.clamp(min=0) if corr > 0 else (-f).clamp(min=0))
    return torch.where(band, r * (1 - fa2) + back, r)


def _solve(r, case, h):
    NY, NX = r.shape
    if case["poisson"] == "periodic":
        kx = 2 * math.pi * torch.fft.rfftfreq(NX, device="cuda", dtype=torch.float64)[None, :]
        ky = 2 * math.pi * torch.fft.fftfreq(NY, device="cuda", dtype=torch.float64)[:, None]
        k2 = kx * kx + ky * ky
        k2[0, 0] = 1.0
        P = -torch.fft.rfft2(r) / k2
        P[0, 0] = 0
        return torch.fft.irfft2(P, s=(NY, NX))
    if case["poisson"] == "cosine":
        # the mirror image's transform; symbol: 0.9 finite differences + 0.1 spectral
        m = torch.cat([r, r.flip(1)], 1)
        m = torch.cat([m, m.flip(0)], 0)
        i = torch.arange(NX + 1, device="cuda", dtype=torch.float64)[None, :]
        j = torch.arange(2 * NY, device="cuda", dtype=torch.float64)[:, None]
        j = torch.minimum(j, 2 * NY - j)
        cx = torch.cos(2 * math.pi / NX * i).float().double()
        cy = torch.cos(2 * math.pi / NY * j).float().double()
        sp = (math.pi / NX * (i + 0.5)).square() + (math.pi / NY * (j + 0.5)).square()
        den = 0.9 * (1 - cx / 2 - cy / 2) + 0.1 * sp
        s = torch.where((i < NX) & (j < NY), -1 / den, torch.zeros_like(den))
        s[0, 0] = 0
        return torch.fft.irfft2(torch.fft.rfft2(m) * s, s=(2 * NY, 2 * NX))[:NY, :NX].contiguous()
    # free space: convolution with the log kernel, its self cell averaged over a disk
    i = torch.arange(2 * NX, device="cuda", dtype=torch.float64)[None, :]
    j = torch.arange(2 * NY, device="cuda", dtype=torch.float64)[:, None]
    d2 = torch.minimum(i, 2 * NX - i).square() + torch.minimum(j, 2 * NY - j).square()
    d2[0, 0] = 1.0
    G = torch.log(h * d2.sqrt()) / (2 * math.pi)
    G[0, 0] = (2 * math.log(h / math.sqrt(math.pi)) - 1) / (4 * math.pi)
    P = torch.fft.rfft2(r, s=(2 * NY, 2 * NX)) * torch.fft.rfft2(G)
    return torch.fft.irfft2(P, s=(2 * NY, 2 * NX))[:NY, :NX].contiguous()


def _advdiff(u, v, dt, h, nu):
    dfac, afac = (nu / h) * (dt / h), -0.5 * dt / h
    out = []
    for a in (u, v):
        e, w, n, s = (_shift(a, 1, 0), _shift(a, -1, 0), _shift(a, 0, 1), _shift(a, 0, -1))
        out.append(a + afac * (u * (e - w) + v * (n - s)) + dfac * (e + w + n + s - 4 * a))
    u1, v1 = out
    NY, NX = u.shape
    corr = (u1[:, -1].sum() - u1[:, 0].sum() + v1[-1].sum() - v1[0].sum()) / (2 * NX + 2 * NY)
    u1[:, 0] += corr
    u1[:, -1] -= corr
    v1[0] += corr
    v1[-1] -= corr
    return u1, v1


def exact(case, seed):
    kind = case["kind"]
    if kind not in ("operators", "solve"):
        return None  # whole steps with bodies: no description short of the program itself
    NX, NY = case["bpdx"] * BS, case["bpdy"] * BS
    h = 1.0 / (BS * max(case["bpdx"], case["bpdy"]))
    if kind == "solve":
        r = _fade(_rhs(NX, NY, h, seed), case, h)
        return dict(p=_solve(r, case, h), rhs=r)
    dt = _dt(case)
    vel = _velocity(NX, NY, h, seed, 0.1)
    u, v = _advdiff(vel[0], vel[1], dt, h, 1e-3)
    r = _fade(_div(u, v) * (0.5 * h / dt), case, h)
    p = _solve(r, case, h)
    fac = -0.5 * dt / h
    return dict(u=u + fac * (_shift(p, 1, 0) - _shift(p, -1, 0)),
                v=v + fac * (_shift(p, 0, 1) - _shift(p, 0, -1)), p=p)
