"""Momenta and fields whose squares leave the range of a float: the push gives
what IEEE square roots and divisions give (em2d/particles.c:1137-1192), a
particle at rest where 1 + u^2 is infinite and no rotation where 1 + t^2 is,
particle by particle bit for bit; and the short square root is checked up to
the largest float."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from em2d_driver import weibel
from test_gpu_parity import gpu_run, matched, oracle_run
from test_gpu_rounding import LIMIT, check

pytestmark = pytest.mark.gpu

# u and B in units in which t = 0.035 B / gamma; squares up to and beyond 2^126, 2^127 and 2^128
U = [1e17, 9e18, 1.2e19, 1.5e19, 1.84e19, 1.9e19, 1e30]
B = [1e17, 2.4e20, 3e20, 4.5e20, 5.2e20, 5.3e20, 1e30]
E = [1e20, 5e20, 1e22]


@pytest.mark.parametrize("species", [1, 2])
@pytest.mark.parametrize("what,value", [("u", v) for v in U] + [("B", v) for v in B] + [("E", v) for v in E])
def test_push_at_extreme_values(gpu, oracle, what, value, species):
    print(f"extremes: {what} {value:g} species {species}", flush=True)
    cfg = weibel(32, 24, 2, uth=0.0 if what == "u" else 0.1)
    cfg["species"] = cfg["species"][:species]
    if what == "u":
        for k, s in enumerate(cfg["species"]):
            s["ufl"] = [value, 0.0, -0.3] if k == 0 else [0.2, value, 0.5 * value]
    else:
        v = [0.6 * value, 0.0, 0.8 * value] if what == "B" else [0.0, value, 0.1]
        cfg["init_fld"] = {f"{what}_0": v, ("E_0" if what == "B" else "B_0"): [0.0, 0.0, 0.1]}
    g, o = gpu_run(gpu, cfg, ids=True), oracle_run(oracle, cfg, ids=True)
    try:
        g.step(1)
        o.step(1)
        for k in range(species):
            pg, po = matched(gpu, oracle, g, o, k)
            for f in pg.dtype.names:
                a, b = pg[f], po[f]
                same = (a == b) | ((a != a) & (b != b))
                assert same.all(), (k, f, a[~same][:3], b[~same][:3])
    finally:
        g.close()
        o.close()


def test_square_root_up_to_the_largest_float(gpu):
    assert check(gpu, LIMIT, 0x7F800000 - LIMIT, 1.0)[1] == 0
