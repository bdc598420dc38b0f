"""The counters that finish a push (zk_spec_finalize_set) and their copy in
page-locked memory: one to four species, with and without a copy, partial
sums fewer and more than a workgroup's threads."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

MAX = 4  # species of one launch
CTR = np.dtype([(n, np.int32) for n in ("np_total", "n_sorted", "n_dead", "n_overflow", "n_slack", "n_unplaced",
                                        "n_overfull", "ovf_sorted", "n_fx_range", "pad")] +
               [("npush", np.uint64), ("energy", np.float64)])


class FinalizeSet(C.Structure):
    _fields_ = [("n", C.c_int), ("ctr", C.c_void_p * MAX), ("probe", C.c_void_p * MAX), ("seq", C.c_uint * MAX),
                ("epart", C.c_void_p * MAX), ("nparts", C.c_int * MAX), ("qm", C.c_double * MAX),
                ("dx0", C.c_double * MAX), ("dx1", C.c_double * MAX)]


@pytest.mark.parametrize("n,nparts", [(1, 1), (1, 1025), (3, 7), (4, 1024), (4, 5000)])
def test_counters_reach_the_host(gpu, n, nparts):
    print(f"probe: {n} species, {nparts} partial sums", flush=True)
    rng = np.random.default_rng(nparts)
    f = FinalizeSet(n=n)
    keep = []
    for k in range(n):
        c = np.zeros(1, CTR)
        c["np_total"], c["n_dead"], c["n_slack"], c["npush"] = 1000 + k, 10 * k, 5, 1 << 40
        c["n_overflow"], c["ovf_sorted"], c["n_fx_range"] = -3 - k, 77, k
        part = np.round(rng.uniform(0, 1000, nparts))  # whole numbers: the order of the sum is free
        d = torch.from_numpy(c.view(np.uint8)).cuda()
        e = torch.from_numpy(part).cuda()
        h = torch.zeros(CTR.itemsize + 8, dtype=torch.uint8, pin_memory=True)
        keep.append((c, part, d, e, h))
        f.ctr[k], f.epart[k], f.nparts[k] = d.data_ptr(), e.data_ptr(), nparts
        f.probe[k] = h.data_ptr() if k != 1 else None
        f.seq[k], f.qm[k], f.dx0[k], f.dx1[k] = 41 + k, -2.0, 0.5, 0.25
    torch.cuda.synchronize()
    assert gpu.zk_spec_finalize_set(C.byref(f), None) == 0
    torch.cuda.synchronize()
    for k, (c, part, d, e, h) in enumerate(keep):
        exp = c.copy()
        exp["energy"] = -2.0 * part.sum() * 0.5 * 0.25
        exp["npush"] += np.uint64(1000 + k - 10 * k - 5)
        got = d.cpu().numpy().view(CTR)
        assert got.tobytes() == exp.tobytes()
        host = h.numpy()
        if k == 1:
            assert not host.any()
        else:
            assert host[:CTR.itemsize].tobytes() == exp.tobytes()
            assert int(host[CTR.itemsize:].view(np.uint32)[0]) == 41 + k
