"""Stream rows read while another thread runs ticks: tests/native/
stream_reads_check.cpp drives libkunhip.so's stream contexts on the CPU."""
import os
import shutil
import subprocess

import pytest

from kunquant_amd.build import CSRC, LIB_DIR
from kunquant_amd.workloads import catalog

HERE = os.path.dirname(os.path.abspath(__file__))
ROCM_LIB = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "lib")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_a_row_is_of_one_tick(tmp_path):
    exe = str(tmp_path / "stream_reads_check")
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-pthread", "-rdynamic", "-I", CSRC,
                    os.path.join(HERE, "native", "stream_reads_check.cpp"), "-o", exe, "-L", LIB_DIR, "-lkunhip", "-ldl",
                    f"-Wl,-rpath,{LIB_DIR}", f"-Wl,-rpath,{ROCM_LIB}", f"-Wl,-rpath-link,{ROCM_LIB}"], check=True)
    r = subprocess.run([exe, "stream_f64", catalog.library_path("stream_f64")], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
