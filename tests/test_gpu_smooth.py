"""Filter passes of one launch (zk_smooth) against the passes one after the
other in numpy float32, guard handling of kernel_x and kernel_y
(em2d/current.c:316-413) included, bit for bit: pass counts at the limits of
each launch shape, grids smaller than the margins, partial last blocks,
moving windows and open y boundaries.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

f32 = np.float32


def x_pass(J, nx, ny, sa, sb, periodic):
    o = J.copy()
    r = J[1:ny + 1]
    o[1:ny + 1, 1:nx + 1] = sa * r[:, 0:nx] + sb * r[:, 1:nx + 1] + sa * r[:, 2:nx + 2]
    if periodic:
        for b in (0, nx + 1, nx + 2):
            o[1:ny + 1, b] = o[1:ny + 1, (b - 1) % nx + 1]
    return o


def y_pass(J, nx, ny, sa, sb, periodic):
    o = J.copy()
    c = J[:, 1:nx + 1]
    o[1:ny + 1, 1:nx + 1] = sa * c[0:ny] + sb * c[1:ny + 1] + sa * c[2:ny + 2]
    if periodic:
        for b in (0, ny + 1, ny + 2):
            o[b] = o[(b - 1) % ny + 1]
    return o


# (nx, ny, x passes, y passes)
CASES = [(3, 3, 1, 0), (97, 61, 3, 3), (62, 13, 1, 1), (63, 6, 1, 2), (70, 5, 0, 2), (40, 9, 2, 6), (33, 10, 16, 7),
         (300, 4, 16, 0), (5, 40, 5, 12), (128, 128, 0, 12), (511, 33, 5, 0)]


@pytest.mark.parametrize("open_y", [0, 1], ids=["periodic_y", "open_y"])
@pytest.mark.parametrize("periodic_x", [1, 0], ids=["periodic_x", "window"])
@pytest.mark.parametrize("nx,ny,n1,n2", CASES)
def test_passes_of_one_launch(gpu, nx, ny, n1, n2, periodic_x, open_y):
    print(f"smooth: {nx}x{ny} x {n1} y {n2} periodic_x {periodic_x} open_y {open_y}", flush=True)
    rng = np.random.default_rng(nx * ny + n1)
    J = rng.standard_normal((ny + 3, nx + 3, 3)).astype(f32)
    # guards of a folded axis are their images
    if periodic_x:
        J = J[:, (np.arange(nx + 3) - 1) % nx + 1]
    if not open_y:
        J = J[(np.arange(ny + 3) - 1) % ny + 1]
    J = np.ascontiguousarray(J)
    sa = rng.uniform(0.1, 0.3, n1 + n2).astype(f32)
    sb = (1 - 2 * sa).astype(f32)
    exp = J
    for p in range(n1 + n2):
        step, per = (x_pass, periodic_x) if p < n1 else (y_pass, not open_y)
        exp = step(exp, nx, ny, sa[p], sb[p], per)
    a = torch.from_numpy(J).cuda()
    b = torch.zeros_like(a)
    torch.cuda.synchronize()
    P = C.POINTER(C.c_float)
    rc = gpu.zk_smooth(C.c_void_p(a.data_ptr()), C.c_void_p(b.data_ptr()), nx, ny, nx + 3, n1, n2,
                       sa.ctypes.data_as(P), sb.ctypes.data_as(P), periodic_x, open_y, None)
    assert rc == 0
    torch.cuda.synchronize()
    assert b.cpu().numpy().tobytes() == exp.tobytes()
