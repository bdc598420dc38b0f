"""The reverse push of a set of species in one launch, against FP64 autograd:
one species, more species than one launch takes, grids whose edge tiles are
cut, grids split over many and over few workgroups a tile, and a loss that
ends before the run does (steps whose adjoints are all zero, so that no
maximum for the fixed-point scale is known until later).

Differentiable runs have no counterpart in the reference.
"""
from __future__ import annotations

import ctypes as C
import os
import sys

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from conftest import ROOT

sys.path.insert(0, os.path.join(ROOT, "oracle"))
import diff64  # noqa: E402

from zpic_amd import _lib  # noqa: E402
from zpic_amd import abi as A  # noqa: E402
from zpic_amd import diff  # noqa: E402

pytestmark = pytest.mark.gpu

_libc = C.CDLL(None)
_libc.calloc.restype = C.c_void_p
_libc.calloc.argtypes = [C.c_size_t, C.c_size_t]

STEPS, DX, DT = 4, 0.1, 0.07


def rel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


# (nx, ny, ppc, species, last loss step); 256 x 192 in 192 tiles of 16 x 16
# takes few workgroups a tile, the small grids the most
CASES = [(32, 32, 2, 1, 4), (40, 27, 2, 5, 4), (33, 48, 1, 4, 2), (256, 192, 1, 2, 4)]


@pytest.mark.parametrize("nx,ny,ppc,ns,last", CASES)
def test_reverse_push_of_a_species_set(nx, ny, ppc, ns, last):
    print(f"adjoint set: {nx}x{ny} ppc {ppc} species {ns} last {last}", flush=True)
    lib = _lib.load()
    diff._declare(lib)
    abi = A.make_abi(True)
    rng = np.random.default_rng(nx + ns)
    n2, box, dt = (C.c_int * 2)(nx, ny), (C.c_float * 2)(nx * DX, ny * DX), C.c_float(DT)
    lib.zpic_rand_clear()
    lib.set_rand_seed(7, 11)
    species = C.cast(_libc.calloc(ns, C.sizeof(abi.t_species)), C.POINTER(abi.t_species))
    for k in range(ns):
        lib.spec_new(C.byref(species[k]), b"s%d" % k, C.c_float(-1.0 - 0.25 * k), (C.c_int * 2)(ppc, ppc),
                     (C.c_float * 3)(0.1 * k, -0.2, 0.6 * (-1) ** k), (C.c_float * 3)(0.1, 0.1, 0.1), n2, box, dt, None)
    sim = abi.t_simulation()
    lib.sim_new(C.byref(sim), n2, box, dt, C.c_float(0.0), 0, species, ns)
    full = np.ctypeslib.as_array(C.cast(sim.emf.B_buf, C.POINTER(C.c_float)), shape=(ny + 3, nx + 3, 3))
    i, j = np.remainder(np.arange(nx + 3) - 1, nx), np.remainder(np.arange(ny + 3) - 1, ny)
    full[:] = (1e-2 * rng.standard_normal((ny, nx, 3))).astype(np.float32)[j][:, i]
    lib.emf_mark_host_dirty(C.byref(sim.emf))
    p0 = [A.particles_view(species[k]).copy() for k in range(ns)]
    d = lib.zpic_diff_new(C.byref(sim), STEPS, 2, 1, last)
    try:
        loss = float(lib.zpic_diff_forward(d))
        dE, dB = (np.zeros((ny + 3, nx + 3, 3), np.float32) for _ in range(2))
        parts = [np.zeros((len(p), 5), np.float32) for p in p0]
        FP = C.POINTER(C.c_float)
        arr = (FP * ns)(*[p.ctypes.data_as(FP) for p in parts])
        lib.zpic_diff_backward(d, dE.ctypes.data_as(FP), dB.ctypes.data_as(FP), arr)

        grid = diff64.Grid(nx, ny, DX, DX, DT)
        sp, leaves = [], []
        for k in range(ns):
            x, y = (torch.tensor(p0[k][c], dtype=torch.float64, requires_grad=True) for c in ("x", "y"))
            u = torch.tensor(np.stack([p0[k][c] for c in ("ux", "uy", "uz")], 1), dtype=torch.float64,
                             requires_grad=True)
            leaves.append((x, y, u))
            sp.append(diff64.Species(float(species[k].q), -1.0 - 0.25 * k, torch.tensor(p0[k]["ix"]),
                                     torch.tensor(p0[k]["iy"]), x, y, u))
        B = torch.tensor(full.astype(np.float64), requires_grad=True)
        E = torch.zeros_like(B, requires_grad=True)
        ref = diff64.run_loss(grid, sp, E, B, STEPS, 1, last)[0]
        ref.backward()
        gp = [torch.cat([x.grad[:, None], y.grad[:, None], u.grad], 1).numpy() for x, y, u in leaves]
        print(f"loss {rel(loss, float(ref.detach())):.1e} dE {rel(dE, E.grad):.1e} dB {rel(dB, B.grad):.1e} "
              f"parts {[f'{rel(a, b):.1e}' for a, b in zip(parts, gp)]}", flush=True)
        # float32 state, weights and sums over a few steps: the bounds of the two-species gradient tests
        assert rel(loss, float(ref.detach())) <= 1e-5
        assert rel(dE, E.grad) <= 1e-4 and rel(dB, B.grad) <= 1e-4
        for a, b in zip(parts, gp):
            assert rel(a, b) <= 1e-4
    finally:
        lib.zpic_diff_delete(d)
        lib.sim_delete(C.byref(sim))
