"""Re-sorts whose scatter scans the tile counts itself (few tiles) and those
with a scan launch (more): where the particles are sorted does not enter their
motion, so a run re-sorted before a step has, after it, the particles of a run
that was not, bit for bit and each once.  Particles that moved to neighbour
tiles and farther, removed ones and the unsorted tail of a moving window, at
the tile counts around the limit.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from em2d_driver import Em2dRun, lwfa, weibel

pytestmark = pytest.mark.gpu


def pair(gpu, cfg, steps, sorts):
    """Particles after `steps` and one more step, without and with re-sorts in
    front of the last."""
    out = []
    for n in (0, sorts):
        r = Em2dRun(gpu, cfg, sync=lambda q: gpu.sim_sync_host(C.byref(q.sim)))
        try:
            r.step(steps)
            for _ in range(n):
                for k in range(len(cfg["species"])):
                    gpu.zpic_spec_sort(C.byref(r.species[k]))
            r.step(1)
            s = r.state()
            out.append([s[f"part{k}"].copy() for k in range(len(cfg["species"]))])
        finally:
            r.close()
    return out


def same(a, b):
    assert len(a) == len(b) > 0
    assert sorted(x.tobytes() for x in a) == sorted(x.tobytes() for x in b)


# 16 x 16 tiles: 1, 6, 255, 256, 257 and 272 of them
@pytest.mark.parametrize("nx,ny", [(16, 16), (40, 33), (255 * 16, 16), (256, 256), (257 * 16, 16), (272, 256)])
@pytest.mark.parametrize("uz", [0.3, 30.0], ids=["near", "far"])
@pytest.mark.parametrize("sorts", [1, 3])
def test_every_particle_once(gpu, nx, ny, uz, sorts):
    print(f"resort: {nx}x{ny} uz {uz} sorts {sorts}", flush=True)
    a, b = pair(gpu, weibel(nx, ny, 1, uz=uz, uth=uz / 3, n_sort=0), 7, sorts)
    for k in range(2):
        assert len(a[k]) == nx * ny
        same(a[k], b[k])


@pytest.mark.parametrize("nx,ny", [(120, 32), (4300, 16)])
@pytest.mark.parametrize("steps", [4, 9])
def test_tail_and_removed_particles(gpu, nx, ny, steps):
    print(f"resort window: {nx}x{ny} after {steps} steps", flush=True)
    (a,), (b,) = pair(gpu, lwfa(nx, ny, start=1.0, smooth_level=1), steps, 1)
    same(a, b)
    assert (b["ix"] >= 0).all() and (b["ix"] < nx).all()
