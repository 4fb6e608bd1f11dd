"""Whole steps with disks on the routes that the other tests leave out: ragged strips with streamed
stores (FP64 planes beyond the cache), at FP32 and with the iterative penalization, and a disk in
the fade band with the cosine solver."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def cylinder(mod, r=0.05, x=0.25, y=0.25, **kw):
    return mod.disk(r, x, y, xvel=0.2, bFixed=True, bForced=True, **kw)


def velocity(sim, seed, scale=0.05):
    return scale * np.random.default_rng(seed).standard_normal((2, sim.NY, sim.NX))


def test_ragged_streamed_stencils(cup, oracle_mod):
    """2912 x 1984: six planes exceed the 256 MB from which stores are streamed, and 96 of the
    last strip's 256 columns are cells.  advDiff cell by cell against the oracle (the boundary
    cells carry a correction summed in another order, within 1e-15 of values below one)."""
    kw = dict(extent=1.0, nu=3e-3, poisson="periodic")  # no transform of this length: stencils only
    g, o = cup.Simulation(91, 62, **kw), oracle_mod.Oracle(91, 62, **kw)
    assert g.NX * g.NY * 48 > 256 << 20 and g.NX % 256 != 0
    vel = velocity(g, 17, 0.3)
    for sim in (g, o):
        sim.set_field(0, vel)
        sim.set_scalars(uinf=(-0.11, 0.07))
        sim.advdiff(1.3e-5)
    a, b = g.get_field(cup.VEL), o.get_field(oracle_mod.VEL)
    inner = (slice(None), slice(1, -1), slice(1, -1))
    assert np.array_equal(a[inner], b[inner]) and np.abs(a - b).max() < 1e-15
    g.close()


@pytest.mark.parametrize("bp,precision", [((91, 62), "fp64"), ((9, 5), "fp64"), ((9, 5), "fp32")])
def test_merged_and_separate_launches_agree(cup, bp, precision):
    """A step's parts in merged launches and (with their timers on) in launches of their own: the
    same bits, on ragged grids whose stores are streamed, are not, and hold float."""
    got = []
    for timed in (False, True):
        sim = cup.Simulation(*bp, extent=1.0, nu=1e-4, CFL=0.1, poisson="freespace",
                             precision=precision, shapes=[cylinder(cup)])
        sim.reset()
        sim.set_field(cup.VEL, velocity(sim, 5))
        if timed:
            sim.timer_enable("advdiff", 16)
        sim.simulate(4)
        if timed:
            assert sim.timer_read("advdiff")[1] == 4
        got.append([sim.get_field(f).tobytes() for f in (cup.VEL, cup.PRES)]
                   + [sorted(sim.shape().items())])
        sim.close()
    assert got[0] == got[1]


def test_ragged_fp32_steps(cup):
    """Ragged whole steps at FP32 against FP64.  A step rounds each velocity about ten times to
    2^-24 of its size: eight steps of that are 5e-6.  The pressure's source is a difference of
    neighbours a hundred times smaller than the values: a hundred times the error."""
    runs = []
    for precision in ("fp64", "fp32"):
        sim = cup.Simulation(9, 5, extent=1.0, nu=1e-4, CFL=0.1, poisson="freespace",
                             precision=precision, shapes=[cylinder(cup)])
        sim.reset()
        sim.simulate(8)
        runs.append((sim.get_field(cup.VEL), sim.get_field(cup.PRES)))
        sim.close()
    (v, p), (v32, p32) = runs
    assert rel(v32, v) < 5e-6 and rel(p32 - p32.mean(), p - p.mean()) < 5e-4


def test_ragged_iterative_steps(cup, oracle_mod):
    """The iterator's kernels on a ragged grid, whole steps against the oracle (the bounds of the
    other whole-step comparisons: 1e-10 for the fields, 1e-8 for the drag)."""
    kw = dict(extent=1.0, nu=1e-3, CFL=0.1, poisson="freespace", iterative_penal=True)
    g = cup.Simulation(9, 4, shapes=[cylinder(cup, 0.08, 0.3, 0.2)], **kw)
    o = oracle_mod.Oracle(9, 4, fs_pad2=False, shapes=[cylinder(oracle_mod, 0.08, 0.3, 0.2)], **kw)
    for sim in (g, o):
        sim.reset()
    for _ in range(4):
        dg, do = g.calc_max_timestep(), o.calc_max_timestep()
        assert abs(dg - do) <= 1e-13 * do
        g.advance(dg)
        o.advance(do)
    assert rel(g.get_field(0), o.get_field(0)) < 1e-10
    assert rel(g.get_field(2), o.get_field(2)) < 1e-10
    a, b = g.shape(), o.shape()
    assert abs(a["drag"] - b["drag"]) <= 1e-8 * abs(b["drag"])


@pytest.mark.parametrize("nsteps", [1, 6])
def test_cosine_disk_in_fade_band(cup, oracle_mod, nsteps):
    """A disk on the walls' blocks with the cosine solver: the obstacle RHS changes the fade factor
    inside the row pass.  Steps against the oracle (bounds as above); the RHS plane after a step is
    the operators' (1e-13: the factor's sums in another order, up to 4096 terms at 16 eps)."""
    shape = dict(r=0.05, x=0.055, y=0.06, yvel=0.05)
    kw = dict(extent=1.0, nu=1e-3, CFL=0.2, poisson="cosine", fadeLen=0.05)
    g, h = (cup.Simulation(8, 4, shapes=[cylinder(cup, **shape)], **kw) for _ in range(2))
    o = oracle_mod.Oracle(8, 4, shapes=[cylinder(oracle_mod, **shape)], **kw)
    for sim in (g, h, o):
        sim.reset()
        sim.set_field(0, velocity(sim, 19))
    for step in range(nsteps):
        dt = o.calc_max_timestep()
        assert abs(g.calc_max_timestep() - dt) <= 1e-13 * dt
        if step == nsteps - 1:  # the last step by operators on a copy of the state
            h.set_field(0, g.get_field(0))
            h.put_objects(dt)
            h.advdiff(dt)
            h.pressure_rhs(dt)
            h.poisson_solve()
        else:
            h.advance(dt)
        g.advance(dt)
        o.advance(dt)
    assert rel(g.get_field(cup.TMP), h.get_field(cup.TMP)) < 1e-13
    assert rel(g.get_field(0), o.get_field(0)) < 1e-10
    assert rel(g.get_field(2), o.get_field(2)) < 1e-10
    a, b = g.shape(), o.shape()
    assert abs(a["drag"] - b["drag"]) <= 1e-8 * max(abs(b["drag"]), abs(b["forcex"]))
