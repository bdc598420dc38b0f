"""spec_time: the GPU's time from the first workgroup of a step's push to the
last of its push, injection and sort, against the times of the same launches
between events (which add a few microseconds each)."""
from __future__ import annotations

import ctypes as C

import pytest

from em2d_driver import Em2dRun, lwfa, weibel
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


def test_all_work_in_one_tile(gpu):
    """147456 particles in the first of 16 tiles: the workgroups of the others
    end long before it."""
    cfg = {"nx": [256, 16], "box": [25.6, 1.6], "dt": 0.07,
           "species": [{"name": "slab", "m_q": -1.0, "ppc": [24, 24], "uth": [0.01] * 3, "n_sort": 0,
                        "density": {"type": "slab", "start": 0.0, "end": 1.6, "n": 1.0}}]}
    phase, kernels = phase_times(gpu, cfg, 2, 8)
    print(f"phase times: one tile spec_time {phase * 1e6:.1f} us, launches {kernels * 1e6:.1f} us", flush=True)
    assert 0.6 * kernels < phase < 1.4 * kernels


def test_every_step_counts(gpu):
    """More phases than the clock has slots, read after every step and not at
    all in between; the field step in the launch that folds the current."""
    r = Em2dRun(gpu, weibel(32, 32, 2), sync=lambda q: gpu.sim_sync_host(C.byref(q.sim)))
    try:
        r.step(1)
        single = []
        for _ in range(60):
            t = gpu.spec_time(), gpu.emf_time()
            r.step(1)
            single.append((gpu.spec_time() - t[0], gpu.emf_time() - t[1]))
        t = gpu.spec_time(), gpu.emf_time()
        r.step(300)
        run = gpu.spec_time() - t[0], gpu.emf_time() - t[1]
        for k, what in enumerate(("spec_time", "emf_time")):
            s = sorted(x[k] for x in single)
            print(f"phase times: {what} {s[0] * 1e6:.2f} to {s[-1] * 1e6:.2f} us a step, "
                  f"{run[k] / 300 * 1e6:.2f} on average over 300", flush=True)
            assert s[0] > 5e-7
            assert 0.5 * s[0] < run[k] / 300 < 2 * s[-1]
    finally:
        r.close()
