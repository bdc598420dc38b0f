"""A particle whose position is not a number crosses no cell edge, as in the
reference, whose ltrim compares (em2d/particles.c:1081-1084): it stays in its
cell, with periodic boundaries, in a moving window and with open y
boundaries, in a tile at the edge of the grid and in one away from it."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from em2d_driver import Em2dRun, weibel

pytestmark = pytest.mark.gpu

FAST = {"uz": 3.0, "uth": 1.0}


@pytest.mark.parametrize("cell", [(40, 37), (18, 1), (63, 63)])
@pytest.mark.parametrize("mode", ["periodic", "one_species", "window", "open_y", "staged"])
def test_nan_particle_stays_in_its_cell(gpu, mode, cell):
    print(f"nan particle: {mode} {cell}", flush=True)
    cfg = {**weibel(80, 64, 2, n_sort=3, **FAST), "moving_window": mode == "window"}
    if mode == "one_species":
        cfg["species"] = cfg["species"][:1]
    gpu.zpic_set_staged_sort(mode == "staged")
    r = Em2dRun(gpu, cfg, sync=lambda q: gpu.sim_sync_host(C.byref(q.sim)))
    try:
        if mode == "open_y":
            gpu.zpic_sim_set_open_y(C.byref(r.sim))
        sp = r.species[0]
        p = next(q for q in (sp.part[i] for i in range(sp.np)) if (q.ix, q.iy) == cell)
        p.x = p.y = float("nan")
        gpu.spec_mark_host_dirty(C.byref(sp))
        for _ in range(7):
            r.step(1)
            s = r.state()
            q = s["part0"][np.isnan(s["part0"]["x"])]
            at = [(int(c["ix"]) + (s["n_move0"] if mode == "window" else 0), int(c["iy"])) for c in q]
            assert at == [cell], at
    finally:
        gpu.zpic_set_staged_sort(0)
        r.close()
