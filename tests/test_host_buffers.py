"""CPU checks of host-side size arithmetic of the library, compiled against its
headers with stand-ins for the HIP calls they make."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")


def run_host_check(name, tmp_path):
    exe = str(tmp_path / name)
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__",
                    "-I" + os.path.join(ROCM, "include"), "-I" + os.path.join(ROOT, "include"),
                    "-I" + os.path.join(ROOT, "regot-python_amd", "csrc"),
                    os.path.join(ROOT, "tests", "host", name + ".cpp"), "-pthread", "-o", exe],
                   check=True, capture_output=True, text=True, timeout=120)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr


needs_gxx = pytest.mark.skipif(shutil.which("g++") is None or
                               not os.path.exists(os.path.join(ROCM, "include", "hip")),
                               reason="needs g++ and the HIP headers")


@needs_gxx
def test_staging_memory_of_wide_problems(tmp_path):
    # n + m values each way, from n + m = 2 up to the largest int sizes
    run_host_check("staging_check", tmp_path)


@needs_gxx
def test_grids_of_wide_problems(tmp_path):
    run_host_check("grid_check", tmp_path)


@needs_gxx
def test_failed_allocations_take_the_handles_spare_memory(tmp_path):
    run_host_check("spare_check", tmp_path)
