"""The benchmark quotes the traffic of the kernel that its forward pass runs.
CPU only."""
import os
import sys

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402


def test_traffic_is_of_the_kernel_that_runs_by_default():
    for path in (bench.KERNEL_SRC, bench.TRAFFIC_FILE):
        assert "k_wide_pair" in open(path).read(), path
