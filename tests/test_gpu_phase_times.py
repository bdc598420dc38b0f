"""spec_time: the GPU's time from the first workgroup of a step's push to the
last of its push, injection and sort, against the times of the same launches
between events (which add a few microseconds each)."""
from __future__ import annotations

import ctypes as C

import pytest

from em2d_driver import Em2dRun, lwfa
from test_gpu_parity import lwfa_with_ions

pytestmark = pytest.mark.gpu


def phase_times(gpu, cfg, warm, steps):
    """spec_time and the push and sort launches' time of `steps` steps, one
    after the other so that neither is timed while the other adds to it."""
    gpu.zpic_kernel_time.restype = C.c_double
    gpu.zpic_kernel_time.argtypes = [C.c_int, C.c_void_p]
    r = Em2dRun(gpu, cfg, sync=lambda q: gpu.sim_sync_host(C.byref(q.sim)))
    try:
        r.step(warm)
        t = gpu.spec_time()
        r.step(steps)
        phase = gpu.spec_time() - t
        gpu.zpic_kernel_timing(1)
        k = [gpu.zpic_kernel_time(c, None) for c in (0, 1)]
        r.step(steps)
        k = [gpu.zpic_kernel_time(c, None) - k[c] for c in (0, 1)]
        return phase, sum(k)
    finally:
        gpu.zpic_kernel_timing(0)
        r.close()


@pytest.mark.parametrize("ions", [0, 1], ids=["one_species", "two_species"])
def test_moving_window_with_an_unsorted_tail(gpu, ions):
    """Between an injection and the next sort the tail is a launch of its own
    behind the fused push of two species."""
    kw = {"nx": 12000, "ny": 32, "dt": 0.01, "start": 0.0}  # a move every fifth step
    phase, kernels = phase_times(gpu, lwfa_with_ions(**kw) if ions else lwfa(**kw), 8, 16)
    print(f"phase times: ions {ions} spec_time {phase * 1e6:.1f} us, launches {kernels * 1e6:.1f} us", flush=True)
    assert 0.6 * kernels < phase < 1.4 * kernels
