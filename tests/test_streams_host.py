"""CPU: the stage order of the adjoint driver and its side streams
(csrc/qbx_internal.h adjoint_dag, csrc/streams.hip), compiled by the host
compiler against a HIP that only keeps book of what is ordered before what
(streams_host.cpp): stages that share an array are ordered, an error at any
stage leaves nothing unordered with the caller's stream, calls at the same time
and captures do not share streams, and the pool of streams is bounded."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "pytential_amd", "csrc")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.mark.skipif(shutil.which("g++") is None or not os.path.isdir(ROCM + "/include/hip"),
                    reason="needs g++ and the HIP headers")
def test_adjoint_stages_and_side_streams(tmp_path):
    exe = str(tmp_path / "streams_host")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I" + ROCM + "/include",
                    "-x", "c++", os.path.join(HERE, "streams_host.cpp"),
                    os.path.join(CSRC, "streams.hip"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
