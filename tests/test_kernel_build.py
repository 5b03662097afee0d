"""Kernels that the build has to hold, from the compiler's remarks it keeps.
CPU only."""
import os

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
