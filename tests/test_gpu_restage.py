"""Reports and uploads of a species whose device buffers were freed and made
again, to track ids or for an adjoint run: the staging buffer they share is
allocated again with them."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from em2d_driver import Em2dRun, weibel

pytestmark = pytest.mark.gpu


def test_charge_after_ids_are_tracked(gpu):
    runs = [Em2dRun(gpu, weibel(24, 16, 2), sync=lambda r: gpu.sim_sync_host(C.byref(r.sim))) for _ in range(2)]
    try:
        for r in runs:
            r.step(3)
        want = runs[0].charge(0)
        # sums of a node's few particles in another order
        near = 32 * 2.0**-23 * np.abs(want).max()
        assert np.abs(runs[1].charge(0) - want).max() <= near
        gpu.spec_track_ids(C.byref(runs[1].species[0]))
        assert np.abs(runs[1].charge(0) - want).max() <= near
        for r in runs:
            r.step(1)  # from the same particles and fields
        a, b = (r.state() for r in runs)
        assert len(a["part0"]) == len(b["part0"])
        assert all(np.array_equal(np.sort(a["part0"][f]), np.sort(b["part0"][f])) for f in ("ux", "uy", "uz"))
    finally:
        for r in runs:
            r.close()
