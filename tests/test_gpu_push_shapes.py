"""The push at the edges of its workgroup shapes: 1024, 512 or 256 threads per
tile by the number of tiles, waves dealt to one, two or three species (the
last unevenly), default and other windows.  Against the oracle: particles
bit-identical after the first push, cells identical and E, B, J within 1e-5
(the bar of every parity test) after six steps without a sort, so that some
particles leave their tiles' windows."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import field_err
from em2d_driver import weibel
from test_gpu_parity import gpu_run, matched, oracle_run

pytestmark = pytest.mark.gpu


def deck(nx, ny, nsp, ppc=1):
    cfg = weibel(nx, ny, ppc, uz=0.6, uth=0.5, n_sort=0, m_q2=-1.0)
    third = dict(cfg["species"][0], name="third", ufl=[0.3, 0.4, 0.0])
    cfg["species"] = (cfg["species"] + [third])[:nsp]
    return cfg


# 256, 272, 512 and 528 tiles of 16 x 16 cells; 7 x 6 tiles of 13 x 11
@pytest.mark.parametrize("nx,ny,nsp", [(256, 256, 1), (256, 256, 3), (272, 256, 2), (512, 256, 1), (512, 256, 3),
                                       (528, 256, 2), (528, 256, 3), (91, 66, 1), (91, 66, 2), (91, 66, 3)])
def test_push_matches_the_oracle(gpu, oracle, nx, ny, nsp):
    cfg = deck(nx, ny, nsp)
    g, o = gpu_run(gpu, cfg, ids=True), oracle_run(oracle, cfg, ids=True)
    try:
        g.step(1)
        o.step(1)
        for k in range(nsp):
            pg, po = matched(gpu, oracle, g, o, k)
            assert pg.tobytes() == po.tobytes()
        g.step(5)
        o.step(5)
        for k in range(nsp):
            pg, po = matched(gpu, oracle, g, o, k)
            assert np.array_equal(pg["ix"], po["ix"]) and np.array_equal(pg["iy"], po["iy"])
        sg, so = g.state(), o.state()
        for f in ("J", "E", "B"):
            assert field_err(sg, so, f) <= 1e-5, f
        assert np.allclose(sg["kin_energy"], so["kin_energy"], rtol=1e-6)
    finally:
        g.close()
        o.close()
