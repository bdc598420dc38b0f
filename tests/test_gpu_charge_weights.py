"""Charge density of weights that a fixed-point sum holds badly or not at all
(em2d/particles.c:1289-1324 adds floats): a particle whose position is not a
number makes the nodes of its cell NaN, and weights many binades below the
particle's charge keep their floats' precision.

Tolerance of the latter: a weight is a product of float32 factors (four
roundings of 2^-24), a node sums at most n of them (2^-24 each), all of one
sign: (4 + n) 2^-24 of the node's own value."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from em2d_driver import Em2dRun, weibel

pytestmark = pytest.mark.gpu

FP = C.POINTER(C.c_float)


def particles_in_cell(gpu, ppc, cell, x, y):
    """A run whose first species has all its particles in one cell."""
    r = Em2dRun(gpu, weibel(32, 24, ppc), sync=lambda q: gpu.sim_sync_host(C.byref(q.sim)))
    sp = r.species[0]
    for i in range(sp.np):
        p = sp.part[i]
        p.ix, p.iy = cell
        p.x, p.y = float(x[i % len(x)]), float(y[i % len(y)])
    gpu.spec_mark_host_dirty(C.byref(sp))
    return r, sp


@pytest.mark.parametrize("cell", [(9, 12), (15, 15), (31, 23)])
def test_small_weights(gpu, cell):
    rng = np.random.default_rng(3)
    x = (10.0 ** rng.uniform(-9, -0.1, 64)).astype(np.float32)
    y = (10.0 ** rng.uniform(-9, -0.1, 61)).astype(np.float32)
    y[::7] = np.float32(1 - 2.0**-24)
    r, sp = particles_in_cell(gpu, 1, cell, x, y)
    try:
        n, q = sp.np, float(sp.q)
        rho = r.charge(0).astype(np.float64)
        wx, wy = (a[np.arange(n) % len(a)].astype(np.float64) for a in (x, y))
        for di, dj, w in ((0, 0, (1 - wx) * (1 - wy)), (1, 0, wx * (1 - wy)), (0, 1, (1 - wx) * wy), (1, 1, wx * wy)):
            want = q * w.sum()
            got = rho[cell[1] + dj, cell[0] + di]
            print(f"charge weights: {cell} corner {di} {dj} {got:.6e} {want:.6e}", flush=True)
            assert abs(got - want) <= (4 + n) * 2.0**-24 * abs(want)
    finally:
        r.close()


def test_tiny_weights_alone(gpu):
    x = np.array([1e-6, 3e-7, 2e-5], np.float32)
    y = np.array([2e-6, 5e-8], np.float32)
    r, sp = particles_in_cell(gpu, 1, (9, 12), x, y)
    try:
        n, q = sp.np, float(sp.q)
        k = np.arange(n)
        want = q * np.sum(x[k % 3].astype(np.float64) * y[k % 2].astype(np.float64))
        got = float(r.charge(0)[13, 10])
        assert abs(got - want) <= (4 + n) * 2.0**-24 * abs(want), (got, want)
    finally:
        r.close()


def test_nan_position_shows(gpu):
    r = Em2dRun(gpu, weibel(32, 24, 2), sync=lambda q: gpu.sim_sync_host(C.byref(q.sim)))
    try:
        want = r.charge(0)
        sp = r.species[0]
        p = next(q for q in (sp.part[i] for i in range(sp.np)) if (q.ix, q.iy) == (17, 9))
        p.x = float("nan")
        gpu.spec_mark_host_dirty(C.byref(sp))
        got = r.charge(0)
        bad = [tuple(b) for b in np.argwhere(np.isnan(got))]
        assert bad == [(9, 17), (9, 18), (10, 17), (10, 18)]
        ok = ~np.isnan(got)
        assert np.abs(got - want)[ok].max() <= 32 * 2.0**-23 * np.abs(want).max()
        out = np.zeros(33 * 25, np.float32)
        assert gpu.spec_deposit_charge_noalloc(C.byref(sp), out.ctypes.data_as(FP)) == 0
        assert np.array_equal(np.isnan(out.reshape(25, 33)), np.isnan(got))
    finally:
        r.close()
