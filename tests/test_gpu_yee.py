"""The field step (zk_yee) against the three half and whole steps of the
reference's emf_advance (em2d/emf.c:500-562, 573-637, 688-698) in numpy
float32, bit for bit, guard cells included: grids of one unit and of several,
partial last units, rows and columns at their edges, moving windows (with
and without the fused shift, :646-676) and open y boundaries (the Mur
condition of the reference's one-dimensional code, em1d/emf.c:379-406).
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

f32 = np.float32


def model(E, B, J, nx, ny, dt, dx, dy, periodic_x, open_y, shift):
    E, B = E.copy(), B.copy()
    E0 = E.copy()
    h = f32(dt) / f32(2)
    dtx2, dty2, dtx, dty = h / f32(dx), h / f32(dy), f32(dt) / f32(dx), f32(dt) / f32(dy)
    mur = (f32(dt) - f32(dy)) / (f32(dt) + f32(dy))

    def bhalf():
        # raw rows and columns [-1, n] are buffer [0, n + 1]
        c, r, u = E[:ny + 2, :nx + 2], E[:ny + 2, 1:nx + 3], E[1:ny + 3, :nx + 2]
        b = B[:ny + 2, :nx + 2]
        b[..., 0] += -dty2 * (u[..., 2] - c[..., 2])
        b[..., 1] += dtx2 * (r[..., 2] - c[..., 2])
        b[..., 2] += -dtx2 * (r[..., 1] - c[..., 1]) + dty2 * (u[..., 0] - c[..., 0])

    bhalf()
    # raw [0, n + 1] is buffer [1, n + 2]
    c, left, d = B[1:, 1:], B[1:, :-1], B[:-1, 1:]
    e, j = E[1:, 1:], J[1:, 1:]
    e[..., 0] += dty * (c[..., 2] - d[..., 2]) - f32(dt) * j[..., 0]
    e[..., 1] += -dtx * (c[..., 2] - left[..., 2]) - f32(dt) * j[..., 1]
    e[..., 2] += (dtx * (c[..., 1] - left[..., 1]) - dty * (c[..., 0] - d[..., 0])) - f32(dt) * j[..., 2]
    if open_y:
        for g, i in ((0, 1), (ny + 1, ny)):
            for q in (0, 2):
                E[g, :, q] = E0[i, :, q] + mur * (E[i, :, q] - E0[g, :, q])
    bhalf()
    for F in (E, B):
        if periodic_x:
            F[:] = F[:, (np.arange(nx + 3) - 1) % nx + 1]
        if not open_y:
            F[:] = F[(np.arange(ny + 3) - 1) % ny + 1]
        if shift:
            F[:, :-1] = F[:, 1:].copy()
            F[:, nx:] = 0
    return E, B


CASES = [(3, 3), (58, 5), (59, 6), (61, 13), (130, 4), (97, 61), (20, 31), (1800, 1200)]
MODES = [(1, 0, 0), (0, 0, 0), (0, 0, 1), (0, 1, 0), (0, 1, 1), (1, 1, 0)]


@pytest.mark.parametrize("periodic_x,open_y,shift", MODES)
@pytest.mark.parametrize("nx,ny", CASES)
def test_field_step(gpu, nx, ny, periodic_x, open_y, shift):
    print(f"yee: {nx}x{ny} periodic_x {periodic_x} open_y {open_y} shift {shift}", flush=True)
    rng = np.random.default_rng(nx * ny)
    F = [rng.standard_normal((ny + 3, nx + 3, 3)).astype(f32) for _ in range(3)]
    dt, dx, dy = 0.07, 0.1, 0.13
    Em, Bm = model(*F, nx, ny, dt, dx, dy, periodic_x, open_y, shift)
    E, B, J = (torch.from_numpy(a).cuda() for a in F)
    Eo, Bo = torch.full_like(E, 7.0), torch.full_like(B, 7.0)
    torch.cuda.synchronize()

    class Stamp(C.Structure):
        _fields_ = [("clk", C.c_void_p), ("slot", C.c_int), ("open", C.c_int)]

    p = [C.c_void_p(t.data_ptr()) for t in (E, B, J, Eo, Bo)]
    rc = gpu.zk_yee(*p, nx, ny, nx + 3, C.c_float(dt), C.c_float(dx), C.c_float(dy), periodic_x, open_y, shift, Stamp(),
                    None)
    assert rc == 0
    torch.cuda.synchronize()
    got = Eo.cpu().numpy(), Bo.cpu().numpy()
    for name, a, b in (("E", got[0], Em), ("B", got[1], Bm)):
        bad = np.argwhere(a != b)
        assert len(bad) == 0, (name, len(bad), bad[:5].tolist())
