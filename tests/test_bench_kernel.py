"""bench.py names the kernel that its launch ran, and quotes measured traffic of that kernel alone."""
import os
import sys

import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402


@pytest.mark.parametrize("lanes,waves,name", [(16, 1, "ias15_row_kernel"), (16, 2, "ias15_row_kernel"),
                                              (8, 1, "ias15_kernel"), (4, 1, "ias15_kernel"),
                                              (1, 1, "ias15_lane_kernel"), (1, 2, "ias15_kernel")])
def test_kernel_of_a_launch(lanes, waves, name):
    assert bench.kernel_name(lanes, waves) == name


def test_traffic_is_of_the_kernel_that_ran():
    for form in ("fp64", "mixed+learned"):
        rows, groups = (bench.measured_traffic("c4", form, 262144, k) for k in ("ias15_row_kernel", "ias15_kernel"))
        assert rows and groups and rows != groups
        assert bench.measured_traffic("c5", form, 1048576, "ias15_lane_kernel")
        assert bench.measured_traffic("c5", form, 1048576, "ias15_row_kernel") is None
    assert bench.measured_traffic("c4", "fp64", 1000, "ias15_row_kernel") is None
    # the workload and form that bench.py reports by default have a profile of their default kernel
    assert bench.measured_traffic("c4", "mixed+learned", bench.CONFIGS["c4"]["n"], bench.kernel_name(16, 2))
