"""The fields the particles see (E and B plus external fields) written by the
field step: E + external in float32 at every node, bit for bit, for uniform
and grid fields, either or both, in the separate field step; and the launch
that also folds the current against the separate ones over a few steps, on a
periodic grid and in a moving window.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from em2d_driver import Em2dRun, lwfa, weibel
from zpic_amd import abi as A

pytestmark = pytest.mark.gpu

f32 = np.float32


class Ext(C.Structure):
    _fields_ = [("out", C.c_void_p * 2), ("grid", C.c_void_p * 2), ("uniform", (C.c_float * 3) * 2)]


class Stamp(C.Structure):
    _fields_ = [("clk", C.c_void_p), ("slot", C.c_int), ("open", C.c_int)]


@pytest.mark.parametrize("periodic_x,open_y", [(1, 0), (0, 0), (0, 1)])
@pytest.mark.parametrize("kinds", [("uniform", None), (None, "grid"), ("grid", "uniform")])
@pytest.mark.parametrize("nx,ny", [(61, 13), (1800, 1200)])
def test_field_step_writes_the_particle_fields(gpu, nx, ny, kinds, periodic_x, open_y):
    print(f"ext step: {nx}x{ny} {kinds} periodic_x {periodic_x} open_y {open_y}", flush=True)
    rng = np.random.default_rng(nx)
    F = [torch.from_numpy(rng.standard_normal((ny + 3, nx + 3, 3)).astype(f32)).cuda() for _ in range(3)]
    grid = [torch.from_numpy(rng.standard_normal((ny + 3, nx + 3, 3)).astype(f32)).cuda() for _ in range(2)]
    new = [[torch.full_like(F[0], 7.0) for _ in range(2)] for _ in range(2)]
    part = [torch.full_like(F[0], 7.0) for _ in range(2)]
    uni = rng.standard_normal((2, 3)).astype(f32)
    x = Ext()
    for k, kind in enumerate(kinds):
        if kind:
            x.out[k] = part[k].data_ptr()
            x.uniform[k][:] = uni[k]
            if kind == "grid":
                x.grid[k] = grid[k].data_ptr()
    torch.cuda.synchronize()
    arg = lambda out: ([C.c_void_p(t.data_ptr()) for t in (*F, *out)] +
                       [nx, ny, nx + 3, C.c_float(0.07), C.c_float(0.1), C.c_float(0.13), periodic_x, open_y])
    assert gpu.zk_yee(*arg(new[0]), 0, Stamp(), None) == 0
    assert gpu.zk_yee_ext(*arg(new[1]), 0, C.byref(x), Stamp(), None) == 0
    assert gpu.zk_yee_ext(*arg(new[1]), 1, C.byref(x), Stamp(), None) != 0  # not with a shift
    torch.cuda.synchronize()
    for k in range(2):
        a, b = new[0][k].cpu().numpy(), new[1][k].cpu().numpy()
        assert a.tobytes() == b.tobytes()
        p = part[k].cpu().numpy()
        if not kinds[k]:
            assert np.all(p == 7)
            continue
        add = grid[k].cpu().numpy() if kinds[k] == "grid" else uni[k]
        assert p.tobytes() == (a + add).astype(f32).tobytes()


def wave(i, dx, j, dy):
    return (0.01 * i * dx, -0.02, 0.3 + 0.1 * math.sin(i * dx + j * dy))


@pytest.mark.parametrize("cfg", [{**weibel(61, 33, 1), "ext_fld": {"E_custom": wave, "B_0": [0.0, 0.1, 0.3]}},
                                 {**lwfa(120, 31, smooth_level=1), "ext_fld": {"B_custom": wave}}],
                         ids=["periodic", "window"])
def test_one_launch_equals_the_separate_ones(gpu, cfg):
    runs = [Em2dRun(gpu, cfg, sync=lambda r: gpu.sim_sync_host(C.byref(r.sim))) for _ in range(2)]
    try:
        for _ in range(7):
            for on, r in enumerate(runs):
                gpu.zpic_kernel_timing(on)
                r.step(1)
            gpu.zpic_kernel_timing(0)
            a, b = runs[0].state(), runs[1].state()
            for f in ("E", "B", "J"):
                assert a[f].tobytes() == b[f].tobytes(), f
            for f in ("E_part_buf", "B_part_buf"):
                pa, pb = (getattr(r.sim.emf.ext_fld, f) for r in runs)
                assert bool(pa) == bool(pb)
                if pa:
                    va, vb = (A.grid_view(p, tuple(cfg["nx"])).copy() for p in (pa, pb))
                    assert va.tobytes() == vb.tobytes(), f
    finally:
        gpu.zpic_kernel_timing(0)
        for r in runs:
            r.close()
