"""Host paths of the library that a GPU run reaches only in part or not
safely (buffers freed and made again), on the CPU: the host sources compiled
with gcc together with tests/host_check.c, which stands in for the GPU
runtime and checks every pointer."""
from __future__ import annotations

import glob
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(ROOT, "zpic_amd", "csrc")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("host") / "host_check")
    # launches that no check makes stay unresolved
    subprocess.run(["gcc", "-O1", "-g", "-std=gnu11", "-ffp-contract=off", "-w", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", f"-I{ROOT}/include", f"-I{CSRC}/host", f"-I{CSRC}/kernels",
                    os.path.join(HERE, "host_check.c"), *sorted(glob.glob(f"{CSRC}/host/*.c")), "-o", exe,
                    "-Wl,--unresolved-symbols=ignore-all", "-no-pie", "-lm", "-lpthread"], check=True)
    return exe


@pytest.mark.parametrize("what", ["staging", "noalloc", "reads", "device", "slab"])
def test_host_path(program, what):
    r = subprocess.run([program, what], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stderr
