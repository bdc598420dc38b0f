"""Fold, filter and field step in one launch against the separate launches
(taken while the kernel timers are on), bit for bit over some steps: E, B, J
and energies, for the pass counts at the limits of its workgroup shapes,
grids of one unit and of several, moving windows, open y boundaries,
external fields, wide margins (three windows a node) and particles fast
enough to leave their windows (overflow grid, its flags and their clearing).
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from em2d_driver import Em2dRun, lwfa, weibel

pytestmark = pytest.mark.gpu


def filt(kind, n, both=True):
    return {"xtype": kind, "xlevel": n, **({"ytype": kind, "ylevel": n} if both else {})}


CASES = {
    "plain": (weibel(32, 32, 2), 0, None),
    "cut": (weibel(61, 17, 1, smooth=filt("binomial", 1)), 0, None),
    "units": (weibel(200, 97, 1, smooth=filt("compensated", 2)), 0, None),
    "five_y": (weibel(40, 33, 2, smooth=filt("compensated", 4)), 0, None),
    "six_y": (weibel(40, 33, 2, smooth=filt("binomial", 6)), 0, None),
    "small": (weibel(9, 7, 2, smooth=filt("binomial", 2)), 0, None),
    "y_only": (weibel(48, 40, 2, smooth={"xtype": "none", "xlevel": 3, "ytype": "binomial", "ylevel": 3}), 0, None),
    "fast": (weibel(48, 48, 2, uz=20.0, uth=8.0, n_sort=9, smooth=filt("binomial", 1)), 0, None),
    "margin": (weibel(64, 48, 2, n_sort=20), 0, (8, 8, 5)),
    "window": (lwfa(200, 32), 0, None),
    "window_open": (lwfa(200, 31, smooth_level=2), 1, None),
    "open_y_pass": ({**lwfa(130, 40), "smooth": filt("binomial", 2)}, 1, None),
    "external": ({**weibel(48, 40, 2), "ext_fld": {"E_0": [0.01, 0.0, 0.0], "B_0": [0.0, 0.0, 0.3]}}, 0, None),
}


@pytest.mark.parametrize("name", CASES)
def test_one_launch_equals_the_separate_ones(gpu, name):
    cfg, open_y, tiling = CASES[name]
    print(f"field step: {name}", flush=True)
    runs = [Em2dRun(gpu, cfg, sync=lambda r: gpu.sim_sync_host(C.byref(r.sim))) for _ in range(2)]
    try:
        for r in runs:
            if open_y:
                gpu.zpic_sim_set_open_y(C.byref(r.sim))
            if tiling:
                gpu.zpic_sim_set_tiling(C.byref(r.sim), *tiling)
        for step in range(14):
            for on, r in enumerate(runs):
                gpu.zpic_kernel_timing(on)
                r.step(1)
            gpu.zpic_kernel_timing(0)
            if step % 3 and step != 13:
                continue
            a, b = runs[0].state(), runs[1].state()
            for f in ("E", "B", "J"):
                assert a[f].tobytes() == b[f].tobytes(), (step, f)
                assert np.any(a[f]) or step < 13, (step, f)  # a window starts without plasma
            assert np.array_equal(a["emf_energy"], b["emf_energy"])
            assert np.allclose(a["kin_energy"], b["kin_energy"], rtol=1e-12)  # FP64 sums of other lengths
    finally:
        gpu.zpic_kernel_timing(0)
        for r in runs:
            r.close()
