"""The planner's validation against the part of the operator table that an evaluation reads
(cxx/validate_main.cpp, compiled with the host planner)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "ddfmm_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_offsets_outside_the_live_table_are_refused(oplib, tmp_path):
    exe = str(tmp_path / "validate")
    srcs = [os.path.join(CSRC, f) for f in ("tree.cpp", "mlib.cpp", "planner.cpp", "tiles.cpp")]
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, os.path.join(HERE, "cxx", "validate_main.cpp"), *srcs,
                    "-o", exe], check=True)
    out = subprocess.run([exe, *oplib], capture_output=True, text=True, timeout=120)
    print(out.stdout, flush=True)
    assert out.returncode == 0, out.stdout + out.stderr
