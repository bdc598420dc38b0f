"""Host-side check of the current reduction's index arithmetic
(zpic_amd/csrc/kernels/reduce_index.h), compiled with g++ from
tests/reduce_index_check.cpp: for odd and even axes, tiles that divide them
or not, margins of 1 to 6 cells, folded or not, the windows that cover each
node, in order, are those of a search over all images and tiles."""
from __future__ import annotations

import json
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
KERNELS = os.path.join(os.path.dirname(HERE), "zpic_amd", "csrc", "kernels")


def test_windows_of_a_node_match_a_plain_search(tmp_path):
    exe = str(tmp_path / "reduce_index_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", f"-I{KERNELS}",
                    os.path.join(HERE, "reduce_index_check.cpp"), "-o", exe], check=True)
    r = json.loads(subprocess.run([exe], check=True, capture_output=True, text=True).stdout.strip())
    assert r["nodes"] > 50_000 and r["bad"] == 0, r
