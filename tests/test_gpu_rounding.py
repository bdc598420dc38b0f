"""The push's short division and square-root sequences against the compiler's
IEEE ones, bit for bit: reciprocal and square root for every float of their
range, quotients by every float of [1, 4) for numerators spread over a
binade (a quotient depends on the numerator's mantissa and the divisor's)."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ONE, FOUR, LIMIT = 0x3F800000, 0x40800000, 0x7E800000  # bit patterns of 1, 4 and 2^126


def check(gpu, first, n, a):
    gpu.zk_rounding_check.argtypes = [C.c_uint, C.c_uint, C.c_float, C.POINTER(C.c_ulonglong)]
    bad = (C.c_ulonglong * 3)()
    assert gpu.zk_rounding_check(first, n, a, bad) == 0
    return list(bad)


def test_reciprocal_and_square_root_of_every_float(gpu):
    for first in range(ONE, LIMIT, 1 << 27):
        n = min(1 << 27, LIMIT - first)
        assert check(gpu, first, n, 1.0)[:2] == [0, 0], hex(first)


def test_quotients(gpu):
    r = np.random.default_rng(5)
    values = [0.035, -0.035, 1.0, 2.0 - 2.0**-23, 1.0 + 2.0**-23, *r.uniform(1.0, 2.0, 64)]
    for a in values:
        assert check(gpu, ONE, FOUR - ONE, float(np.float32(a)))[2] == 0, a
