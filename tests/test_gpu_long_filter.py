"""Current filters of more passes than one launch takes (16 along x, 12 along
y): J after current_update against the passes one after the other in numpy
float32, kernel_x and kernel_y with their guard handling
(em2d/current.c:316-459), bit for bit with the guard columns, and the fields
that the field step makes from it."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from em2d_driver import Em2dRun, weibel
from test_gpu_smooth import x_pass, y_pass
from test_gpu_yee import model

pytestmark = pytest.mark.gpu

f32 = np.float32


def weights(kind, level):
    """(sa, sb) of each pass along an axis (em2d/current.c:297-304, 427-459)"""
    if kind == "none":
        return []
    w = [(f32(0.25), f32(0.5))] * level
    if kind == "compensated":
        a, b = f32(-1), f32((4.0 + 2.0 * level) / level)
        total = f32(2) * a + b
        w = w + [(a / total, b / total)]
    return w


# the y passes follow xlevel; 12 along y end in one launch
CASES = [("none", "binomial", 12), ("none", "binomial", 13), ("none", "compensated", 12), ("binomial", "binomial", 13),
         ("compensated", "compensated", 12), ("binomial", "none", 17), ("compensated", "binomial", 25)]


@pytest.mark.parametrize("open_y", [0, 1], ids=["periodic_y", "open_y"])
@pytest.mark.parametrize("window", [0, 1], ids=["periodic_x", "window"])
@pytest.mark.parametrize("xtype,ytype,level", CASES)
def test_many_passes(gpu, xtype, ytype, level, window, open_y):
    print(f"long filter: x {xtype} y {ytype} level {level} window {window} open_y {open_y}", flush=True)
    nx, ny = 20, 17
    plain = {**weibel(nx, ny, 2), "moving_window": bool(window)}
    filtered = {**plain, "smooth": {"xtype": xtype, "ytype": ytype, "xlevel": level, "ylevel": level}}
    runs = [Em2dRun(gpu, c, sync=lambda r: gpu.sim_sync_host(C.byref(r.sim))) for c in (plain, filtered)]
    try:
        for r in runs:
            if open_y:
                gpu.zpic_sim_set_open_y(C.byref(r.sim))
            r.step(1)  # 0.07 of a cell width of 0.1: the window does not move
        J = runs[0].state()["J"]
        assert np.any(J)
        for sa, sb in weights(xtype, level):
            J = x_pass(J, nx, ny, sa, sb, not window)
        for sa, sb in weights(ytype, level):
            J = y_pass(J, nx, ny, sa, sb, not open_y)
        s = runs[1].state()
        bad = np.argwhere(s["J"] != J)
        assert len(bad) == 0, (len(bad), bad[:5].tolist())
        e = runs[1].sim.emf
        E, B = model(np.zeros_like(J), np.zeros_like(J), J, nx, ny, plain["dt"], e.dx[0], e.dx[1], not window, open_y, 0)
        assert np.array_equal(s["E"], E) and np.array_equal(s["B"], B)
    finally:
        for r in runs:
            r.close()
