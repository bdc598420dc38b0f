"""Steps without a deposit, whose fold is left out once J is zero: the field
step is that of zero current, J reads as zero, and deposits before and after
are seen, with and without filter passes, and with a species that has no
particles."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from em2d_driver import Em2dRun, lwfa, weibel
from test_gpu_yee import model

pytestmark = pytest.mark.gpu

FILTER = {"xtype": "compensated", "ytype": "compensated", "xlevel": 1, "ylevel": 1}
CASES = {"plain": weibel(33, 20, 1), "filtered": weibel(48, 32, 1, smooth=FILTER),
         "laser": {**lwfa(90, 20, smooth_level=1), "moving_window": False}}  # the plasma begins beyond the box


@pytest.mark.parametrize("name", CASES)
@pytest.mark.parametrize("n", [0, 2])
def test_steps_without_a_deposit(gpu, name, n):
    print(f"idle current: {name}, {n} steps first", flush=True)
    cfg = CASES[name]
    nx, ny = cfg["nx"]
    r = Em2dRun(gpu, cfg, sync=lambda q: gpu.sim_sync_host(C.byref(q.sim)))
    emf, cur = C.byref(r.sim.emf), C.byref(r.sim.current)
    try:
        r.step(n)
        for k in range(3):
            s = r.state()
            dx, dy = r.sim.emf.dx[0], r.sim.emf.dx[1]
            gpu.current_zero(cur)
            gpu.current_update(cur)
            gpu.emf_advance(emf, cur)
            t = r.state()
            assert not np.any(t["J"]), k
            E, B = model(s["E"], s["B"], np.zeros_like(s["E"]), nx, ny, cfg["dt"], dx, dy, 1, 0, 0)
            assert np.array_equal(t["E"], E) and np.array_equal(t["B"], B), k
        r.step(1)
        assert np.any(r.state()["J"]) == (name != "laser")
    finally:
        r.close()
