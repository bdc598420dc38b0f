"""The reverse of the field step (zk_adj_fields) against the step itself
(zk_yee): the field step is linear, so <lE', E'> + <lB', B'> over its outputs
equals <lE, E> + <lB, B> + <lJ, J> over its inputs; the loss term and the
adjoint of the periodic fold against numpy.  Grids below and above the limits
of the register form, one unit and several.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

f32 = np.float32


class Stamp(C.Structure):
    _fields_ = [("clk", C.c_void_p), ("slot", C.c_int), ("open", C.c_int)]


@pytest.mark.parametrize("nx,ny", [(1, 1), (2, 5), (7, 2), (3, 3), (4, 4), (58, 6), (59, 7), (130, 40), (256, 100)])
def test_transpose_of_the_field_step(gpu, nx, ny):
    print(f"adjoint fields: {nx}x{ny}", flush=True)
    rng = np.random.default_rng(nx * 1000 + ny)
    shape = (ny + 3, nx + 3, 3)
    dev = lambda: torch.from_numpy(rng.standard_normal(shape).astype(f32)).cuda()
    E, B, J, lEo, lBo, F = (dev() for _ in range(6))
    Eo, Bo, lE, lB, lJ, lam, lE2, lB2, lJ2, lam2 = (torch.full_like(E, 7.0) for _ in range(10))
    dt, dx, dy, scale = 0.07, 0.1, 0.13, 0.3
    p = lambda *t: [C.c_void_p(a.data_ptr()) for a in t]
    k = [nx, ny, nx + 3, C.c_float(dt), C.c_float(dx), C.c_float(dy)]
    torch.cuda.synchronize()
    assert gpu.zk_yee(*p(E, B, J, Eo, Bo), *k, 1, 0, 0, Stamp(), None) == 0
    assert gpu.zk_adj_fields(*p(lEo, lBo), None, C.c_float(0), *p(lE, lB, lJ, lam), *k, None) == 0
    torch.cuda.synchronize()
    dot = lambda a, b: float((a.double() * b.double()).sum())
    lhs = dot(lEo, Eo) + dot(lBo, Bo)
    rhs = dot(lE, E) + dot(lB, B) + dot(lJ, J)
    # float32 outputs of a few operations each on both sides: 2^-20 of the sum of magnitudes
    size = float(sum((a.double() * b.double()).abs().sum() for a, b in ((lEo, Eo), (lBo, Bo), (lE, E), (lB, B))))
    assert abs(lhs - rhs) <= 2.0**-20 * size, (lhs, rhs)
    # every raw node takes the adjoints of all nodes with its image
    i, j = np.remainder(np.arange(nx + 3) - 1, nx), np.remainder(np.arange(ny + 3) - 1, ny)
    s = np.zeros((ny, nx, 3))
    np.add.at(s, (j[:, None], i[None, :]), lJ.cpu().numpy().astype(np.float64))
    assert np.allclose(lam.cpu().numpy(), s[j][:, i], rtol=0, atol=2.0**-20 * np.abs(lJ.cpu().numpy()).max() * 16)
    # the loss term is added to the interior of lB before everything else
    lBf = lBo.cpu().numpy()
    lBf[1:ny + 1, 1:nx + 1] += f32(scale) * F.cpu().numpy()[1:ny + 1, 1:nx + 1]
    lBf = torch.from_numpy(lBf).cuda()
    torch.cuda.synchronize()
    assert gpu.zk_adj_fields(*p(lEo, lBo, F), C.c_float(scale), *p(lE, lB, lJ, lam), *k, None) == 0
    assert gpu.zk_adj_fields(*p(lEo, lBf), None, C.c_float(0), *p(lE2, lB2, lJ2, lam2), *k, None) == 0
    torch.cuda.synchronize()
    for a, b in ((lE, lE2), (lB, lB2), (lJ, lJ2), (lam, lam2)):
        assert np.array_equal(a.cpu().numpy(), b.cpu().numpy())
