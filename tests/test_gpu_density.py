"""Charge density and phase space of a species where their kernels change
form, against float64 sums over the same particles (the reference's bins and
weights, em2d/particles.c:1289-1324, 1569-1632).

Tolerance: every weight is a product of float32 factors (a few roundings,
each 2^-24 relative), bin coordinates are float32 values up to the bin count
(an absolute error of bins * 2^-23 in a weight), and the sums add at most
2^-24 of a node per addition; relative to the largest node that is below
(8 + bins + additions) * 2^-23, with the additions per accumulator bounded
by the particles in the largest node."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def deposit(a, b, na, nb, q):
    out = np.zeros((nb, na))
    ia, ib = np.trunc(a).astype(int), np.trunc(b).astype(int)
    wa, wb = a - ia, b - ib
    for oa, ob, w in ((0, 0, (1 - wa) * (1 - wb)), (1, 0, wa * (1 - wb)), (0, 1, (1 - wa) * wb), (1, 1, wa * wb)):
        ok = (ia + oa >= 0) & (ia + oa < na) & (ib + ob >= 0) & (ib + ob < nb)
        np.add.at(out, ((ib + ob)[ok], (ia + oa)[ok]), q * w[ok])
    return out


def simulation(nx, ny, ppc, steps, **kw):
    from zpic_amd import em2d

    sp = em2d.Species("electrons", -1.0, [ppc, ppc], ufl=[0.3, -0.2, 0.1], uth=[0.3] * 3, n_sort=0, **kw)
    sim = em2d.Simulation([nx, ny], [0.1 * nx, 0.1 * ny], 0.07, species=sp)
    for _ in range(steps):
        sim.iter()
    return sim, sp


# one tile, an odd grid with narrow last tiles, tiles split over workgroups or
# not; after 6 steps without a sort some particles are outside their windows
@pytest.mark.parametrize("nx,ny,ppc,steps", [(8, 8, 3, 1), (33, 47, 3, 6), (128, 64, 2, 6), (640, 512, 1, 3)])
def test_charge(nx, ny, ppc, steps):
    sim, sp = simulation(nx, ny, ppc, steps)
    rho = sp.charge().astype(np.float64)
    p = sp.particles
    want = deposit(p["ix"] + p["x"].astype(np.float64), p["iy"] + p["y"].astype(np.float64), nx + 1, ny + 1,
                   -1.0 / ppc**2)
    want[:, 0] += want[:, nx]
    want[0] += want[ny]
    want = want[:ny, :nx]
    assert np.abs(rho - want).max() <= (8 + 16 * ppc**2) * 2.0**-23 * np.abs(want).max()
    sim.close()


# runs of 16384 bins: less than one, exactly one, one and a bit, the most the
# LDS path takes (16), and beyond it
@pytest.mark.parametrize("bins", [(7, 5), (128, 128), (129, 128), (512, 512), (513, 520)])
def test_phase_space(bins):
    nx, ny, ppc = 96, 80, 3
    sim, sp = simulation(nx, ny, ppc, 4)
    (na, nb), rng = bins, [[0.0, 0.1 * nx], [-1.5, 1.5]]
    got = sp.phasespace(["x1", "u3"], [na, nb], rng).astype(np.float64)
    p, f = sp.particles, np.float64
    x = (p["x"].astype(f) + p["ix"]) * f(np.float32(0.1 * nx) / np.float32(nx))
    lo = [f(np.float32(r[0])) for r in rng]
    ra, rb = (n / (f(np.float32(r[1])) - a) for n, r, a in zip((na, nb), rng, lo))
    want = deposit((x - lo[0]) * ra + 0.5, (p["uz"].astype(f) - lo[1]) * rb + 0.5, na, nb, -1.0 / ppc**2)
    most = np.abs(want).max()
    assert np.abs(got - want).max() <= (8 + max(na, nb) + most * ppc**2) * 2.0**-23 * max(most, 1.0 / ppc**2)
    sim.close()
