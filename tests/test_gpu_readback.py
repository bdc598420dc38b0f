"""Reads of device memory into ordinary host memory (zpic_d2h): sizes around
the chunk limits of the staged path, with and without a live simulation to
hold its chunks, and two threads at once (one finds the chunks taken)."""
from __future__ import annotations

import ctypes as C
import threading

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from zpic_amd import em2d

pytestmark = pytest.mark.gpu

MIB = 1 << 20
SIZES = [4, 8 * MIB - 4, 8 * MIB, 8 * MIB + 4, 13 * MIB + 12, 16 * MIB, 16 * MIB + 4, 37 * MIB + 20]


def read(gpu, src, nbytes):
    out = np.full(nbytes // 4 + 2, -1, np.int32)
    gpu.zpic_d2h(C.c_void_p(out.ctypes.data + 4), C.c_void_p(src.data_ptr()), C.c_size_t(nbytes))
    assert out[0] == -1 and out[-1] == -1
    return out[1:-1]


@pytest.mark.parametrize("held", [True, False], ids=["simulation", "none"])
@pytest.mark.parametrize("nbytes", SIZES)
def test_sizes(gpu, nbytes, held):
    print(f"readback: {nbytes} bytes, held {held}", flush=True)
    sim = em2d.Simulation([16, 16], [1.6, 1.6], 0.05) if held else None
    a = torch.arange(nbytes // 4, dtype=torch.int32, device="cuda") * 3 - 7
    torch.cuda.synchronize()
    for _ in range(2):
        assert (read(gpu, a, nbytes) == a.cpu().numpy()).all()
    del sim


def test_two_threads(gpu):
    sim = em2d.Simulation([16, 16], [1.6, 1.6], 0.05)
    src = [torch.arange(k, k + 5 * MIB, dtype=torch.int32, device="cuda") for k in range(2)]
    torch.cuda.synchronize()
    ok = [0, 0]

    def work(k):
        ref = src[k].cpu().numpy()
        for _ in range(8):
            ok[k] += bool((read(gpu, src[k], 20 * MIB) == ref).all())

    th = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    [t.start() for t in th]
    [t.join() for t in th]
    assert ok == [8, 8]
    del sim
