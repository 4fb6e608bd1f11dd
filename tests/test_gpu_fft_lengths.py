"""Poisson solves at every transform length and at ragged free-space sizes against 64-bit
references (numpy / scipy FFTs of the same operators, not the library's transforms).

Tolerance: the right-hand side is white noise, so every mode carries the same weight and the
symbol scales signal and rounding alike.  A transform of 2^m points loses at most 4 eps per
radix-2 level (a product and two sums per level, each within eps of its operands); a solve and its
reference each pass at most 4 transforms of 13 levels: 2 * 4 * 13 * 4 eps = 9.2e-14."""
import numpy as np
import pytest
from scipy.fft import dctn, idctn

pytestmark = pytest.mark.gpu

TOL = 2 * 4 * 13 * 4 * np.finfo(np.float64).eps


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def solve(cup, poisson, bpdx, bpdy, seed):
    sim = cup.Simulation(bpdx, bpdy, extent=1.0, nu=1e-3, fadeLen=0.0, poisson=poisson)
    r = np.random.default_rng(seed).normal(size=(32 * bpdy, 32 * bpdx))
    if poisson != "freespace":
        r -= r.mean()
    p = sim.poisson_dense(r)
    h = sim.scalars()["h"]
    sim.close()
    return r, p, h


@pytest.mark.parametrize("bpdx,bpdy", [(1, 128), (2, 64), (4, 32), (8, 16), (16, 8), (32, 4),
                                       (64, 2), (128, 1), (256, 1)])
def test_periodic_lengths(cup, bpdx, bpdy):
    r, p, _ = solve(cup, "periodic", bpdx, bpdy, 1)
    NY, NX = r.shape
    kx = 2 * np.pi * np.fft.rfftfreq(NX)[None, :]
    ky = 2 * np.pi * np.fft.fftfreq(NY)[:, None]
    k2 = kx * kx + ky * ky
    k2[0, 0] = 1
    P = -np.fft.rfft2(r) / k2
    P[0, 0] = 0
    assert rel(p, np.fft.irfft2(P, s=r.shape)) < TOL


@pytest.mark.parametrize("bpdx,bpdy", [(1, 64), (2, 32), (4, 16), (8, 8), (16, 4), (32, 2),
                                       (64, 1), (128, 1), (1, 1)])
def test_cosine_lengths(cup, bpdx, bpdy):
    r, p, _ = solve(cup, "cosine", bpdx, bpdy, 2)
    NY, NX = r.shape
    i, j = np.arange(NX)[None, :], np.arange(NY)[:, None]
    cx = np.cos(np.pi / NX * 2.0 * i).astype(np.float32).astype(np.float64)
    cy = np.cos(np.pi / NY * 2.0 * j).astype(np.float32).astype(np.float64)
    sp = (np.pi / NX * (i + 0.5)) ** 2 + (np.pi / NY * (j + 0.5)) ** 2
    s = -1 / (0.9 * (1 - cx / 2 - cy / 2) + 0.1 * sp)
    s[0, 0] = 0
    assert rel(p, idctn(s * dctn(r, type=2), type=2)) < TOL


@pytest.mark.parametrize("bpdx,bpdy", [(1, 1), (1, 64), (2, 33), (3, 17), (5, 9), (9, 5), (17, 3),
                                       (33, 2), (65, 1), (128, 1), (125, 2)])
def test_freespace_lengths(cup, bpdx, bpdy):
    r, p, h = solve(cup, "freespace", bpdx, bpdy, 3)
    NY, NX = r.shape
    i, j = np.arange(2 * NX)[None, :], np.arange(2 * NY)[:, None]
    d2 = (np.minimum(i, 2 * NX - i) ** 2 + np.minimum(j, 2 * NY - j) ** 2).astype(np.float64)
    d2[0, 0] = 1
    G = np.log(h * np.sqrt(d2)) / (2 * np.pi)
    G[0, 0] = (2 * np.log(h / np.sqrt(np.pi)) - 1) / (4 * np.pi)
    P = np.fft.rfft2(r, s=G.shape) * np.fft.rfft2(G)
    assert rel(p, np.fft.irfft2(P, s=G.shape)[:NY, :NX]) < TOL


def test_cosine_step_leaves_whole_rhs(cup):
    """A whole step with the cosine solver forms the right-hand side inside the row pass; the
    RHS plane afterwards holds it on every cell (faded), as the operators leave it.  Both form
    the same cells with the same operations; only the fade factor's sums may differ by rounding:
    a relative 1e-13 covers 4096-term sums at 16 eps."""
    kw = dict(extent=1.0, nu=1e-3, fadeLen=0.05, poisson="cosine")
    d = cup.disk(0.06, 0.4, 0.25, xvel=0.2, bFixed=True, bForced=True)
    a, b = (cup.Simulation(16, 8, shapes=[d], **kw) for _ in range(2))
    for s in (a, b):
        s.reset()
        s.simulate(3)
    dt = a.calc_max_timestep()
    a.advance(dt)
    b.put_objects(dt)
    b.advdiff(dt)
    b.pressure_rhs(dt)
    b.poisson_solve()
    ra, rb = a.get_field(cup.TMP), b.get_field(cup.TMP)
    assert rel(ra, rb) < 1e-13 and rel(a.get_field(cup.PRES), b.get_field(cup.PRES)) < TOL


def test_cosine_fade_repeatable(cup):
    """The row pass fades the band cells in place: the same right-hand side gives the same
    solution and the same faded plane every time."""
    sim = cup.Simulation(64, 8, extent=1.0, nu=1e-3, fadeLen=0.02, poisson="cosine")
    r = np.random.default_rng(5).normal(size=(256, 2048))
    got = set()
    for _ in range(20):
        sim.set_field(cup.TMP, r)
        sim.poisson_solve()
        got.add((sim.get_field(cup.TMP).tobytes(), sim.get_field(cup.PRES).tobytes()))
    assert len(got) == 1
