"""The kernels that take several fine steps per launch give results that do not
depend on the order in which a workgroup's threads run between two barriers:
a CPU build of csrc/steps.hip (tests/cpu) runs every mode, tile and number of
steps with the threads in ascending and in descending order."""
import os
import subprocess

import pytest

from acoustic_isotropic_operators_amd import build

CLANG = "/opt/rocm/llvm/bin/clang++"
HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpu")


def test_results_do_not_depend_on_the_order_of_the_threads(tmp_path):
    if not os.path.exists(CLANG):
        pytest.skip("no clang++ for the CPU build")
    exe = str(tmp_path / "steps_schedule")
    subprocess.run([CLANG, "-x", "c++", "-std=c++17", "-O1", "-ffp-contract=off", "-w", "-I" + HERE, "-I" + build.CSRC,
                    os.path.join(HERE, "steps_schedule.cpp"), "-o", exe], check=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout
