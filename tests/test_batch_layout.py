"""Dependencies and shared memory of batch runs: tests/native/
batch_layout_check.cpp follows the plans that libkunhip.so makes for every
built module, on the CPU."""
import os
import shutil
import subprocess

import pytest

from kunquant_amd.build import CSRC, LIB_DIR
from kunquant_amd.workloads import catalog

HERE = os.path.dirname(os.path.abspath(__file__))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


@pytest.fixture(scope="module")
def follow_plans(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("layout") / "batch_layout_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROCM, "include"), "-I", CSRC,
                    os.path.join(HERE, "native", "batch_layout_check.cpp"), "-o", exe, "-L", LIB_DIR, "-lkunhip",
                    "-L", os.path.join(ROCM, "lib"), "-lamdhip64", "-ldl",
                    f"-Wl,-rpath,{LIB_DIR}", f"-Wl,-rpath,{os.path.join(ROCM, 'lib')}"], check=True)
    return exe


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
@pytest.mark.parametrize("names", [["generic_pair_f32", "generic_f32", "generic_f64_sts"], None])
def test_values_outlive_their_readers(follow_plans, names):
    args = [x for n in (names or catalog.CATALOG) for x in (n, catalog.library_path(n))]
    r = subprocess.run([follow_plans] + args, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-4000:] + r.stderr[-2000:]
    assert int(r.stdout.split()[-2]) >= 9
