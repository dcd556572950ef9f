"""The LDS that the sphere form's plane kernels ask for covers every byte that
their wave exchanges read, lanes without a line included: every pair of
compiled line lengths, 4 to 12 waves and few kept columns, every square length
with every number of columns, both precisions (tests/c_abi/lds_reach.hip,
host code compiled on the spot)."""
import os
import shutil
import subprocess

import pytest

from .util import say

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_exchanges_stay_in_the_blocks_lds(tmp_path):
    exe = str(tmp_path / "lds_reach")
    subprocess.run([HIPCC, "--offload-host-only", "-std=c++17", "-O1", "-w",
                    "-I", os.path.join(ROOT, "letzelphc_amd", "csrc"),
                    "-I", os.path.join(ROOT, "include"),
                    os.path.join(ROOT, "tests", "c_abi", "lds_reach.hip"), "-o", exe], check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True).stdout.split()
    cases, short = int(out[0]), int(out[1])
    say(f"case: LDS of {cases} plane blocks")
    assert cases > 100000 and short == 0
