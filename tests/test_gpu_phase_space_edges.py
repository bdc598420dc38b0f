"""Phase space whose fast axis leaves out part of the particles: those just
below a range and just above it give the edge bins their share and nothing
else, in each form of the kernel (the bins of one LDS copy, several runs of
bins, straight into the grid), against float64 sums; the tolerance is that of
test_gpu_density."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_density import deposit, simulation

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bins", [(40, 30), (200, 200), (513, 520)])
def test_particles_beyond_the_range(bins):
    nx, ny, ppc = 64, 48, 3
    (na, nb), rng = bins, [[0.1, 0.5], [0.2, 0.1 * ny - 0.3]]  # u1 is 0.3 +- 0.3
    sim, sp = simulation(nx, ny, ppc, 2)
    got = sp.phasespace(["u1", "x2"], [na, nb], rng).astype(np.float64)
    p, f = sp.particles, np.float64
    y = (p["y"].astype(f) + p["iy"]) * f(np.float32(0.1 * ny) / np.float32(ny))
    lo = [f(np.float32(r[0])) for r in rng]
    ra, rb = (n / (f(np.float32(r[1])) - a) for n, r, a in zip((na, nb), rng, lo))
    want = deposit((p["ux"].astype(f) - lo[0]) * ra + 0.5, (y - lo[1]) * rb + 0.5, na, nb, -1.0 / ppc**2)
    most = np.abs(want).max()
    assert np.count_nonzero(want[0]) and np.count_nonzero(want[:, 0]) and np.count_nonzero(want[:, -1])
    assert np.abs(got - want).max() <= (8 + max(na, nb) + most * ppc**2) * 2.0**-23 * max(most, 1.0 / ppc**2)
    sim.close()
