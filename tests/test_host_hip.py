"""libkunhip.so on the CPU, its HIP calls answered by host memory
(tests/native/host_hip.hpp): what the runtime does around its kernels."""
import os
import shutil
import subprocess

import pytest

from kunquant_amd.build import CSRC, LIB_DIR
from kunquant_amd.workloads import catalog

HERE = os.path.dirname(os.path.abspath(__file__))
ROCM_LIB = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "lib")
pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")


def _run(tmp_path, name, *args):
    exe = str(tmp_path / name)
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-pthread", "-rdynamic", "-I", CSRC,
                    os.path.join(HERE, "native", name + ".cpp"), "-o", exe, "-L", LIB_DIR, "-lkunhip", "-ldl",
                    f"-Wl,-rpath,{LIB_DIR}", f"-Wl,-rpath,{ROCM_LIB}", f"-Wl,-rpath-link,{ROCM_LIB}"], check=True)
    r = subprocess.run([exe, *args], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr


def test_a_row_is_of_one_tick(tmp_path):
    """Stream rows read while another thread runs ticks."""
    _run(tmp_path, "stream_reads_check", "stream_f64", catalog.library_path("stream_f64"))


def test_corr_takes_the_memory_there_is(tmp_path):
    """corrWith with little device memory free, and what it keeps."""
    _run(tmp_path, "corr_memory_check")
