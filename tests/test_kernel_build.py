"""Kernels that the build has to hold, from the compiler's remarks it keeps of
every file of kernels (tests/test_kernel_resources.py reads their spills).
CPU only."""
import os
import re

import pytest

from acoustic_isotropic_operators_amd import build


def _remarks():
    if not os.path.exists(build.RESOURCE_USAGE):
        pytest.skip("libaiso.so not built here (no resource-usage remarks)")
    return open(build.RESOURCE_USAGE).read()


@pytest.mark.parametrize("kernel", ["13k_ext_ss_tileILi10E", "18k_tomo_adj_ss_tileILi10E"])
def test_tiled_secondary_sources_of_13_to_21_offsets(kernel):
    """Grids of 2^30 points and more take them: the kernels with four z-points
    per lane address a slice with 32-bit byte offsets."""
    assert f"Function Name: _ZN4aiso{kernel}" in _remarks()


# the adjoint step of the velocity gradient on its largest tile, the lockstep
# Born pair, the imaging of 21 offsets
@pytest.mark.parametrize("kernel", [
    "7k_stepsILi64ELi64ELi3ELi1024ELi2ELj16657EE", "11k_wide_pairILi64ELi2ELb0EE", "12k_offset_imgILi10ELi7EE"])
def test_remarks_of_every_file_of_kernels(kernel):
    assert kernel in _remarks()


def test_local_memory_fits_a_workgroup():
    text = _remarks()
    lds = [int(n) for n in re.findall(r"LDS Size \[bytes/block\]: (\d+)", text)]
    assert lds and max(lds) <= 160 << 10
