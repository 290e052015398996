"""The bytes bench.py prices a launch at: every array the right-hand side
kernel reads or writes in the four stages of a step, in bytes per DOF, and
none that it does not.  u^n enters stages 1 to 3 only: the running sum of
stage 4 is acc + dt b_4 k_4."""
import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
import bench  # noqa: E402


@pytest.mark.parametrize("p", [1, 4, 5])
@pytest.mark.parametrize("mixed", [False, True])
def test_launch_bytes_are_the_arrays_of_each_stage(p, mixed):
    w = 4 if mixed else 8
    ff = 6 * (p + 1) ** 2 * w / (p + 1) ** 3
    stages = [
        [w, ff, 8 if mixed else 0, 8, w],        # U_1 (FP64: u^n itself), FF, u^n; running sum, U_2
        [w, ff, 8, 8, 8, w],                     # U_2, FF, u^n, running sum; running sum, U_3
        [w, ff, 8, 8, 8, w],
        [w, ff, 8, 8, 4 if mixed else 0],        # U_4, FF, running sum; running sum, (FP32 copy of u^{n+1})
    ]
    grad, rhs = bench.launch_bytes(1000, mixed, p)
    assert abs(rhs - 1000 * sum(map(sum, stages)) / 4) < 1e-9
    assert abs(grad - 1000 * (w + ff)) < 1e-9


def test_measured_traffic_covers_the_launch_bytes():
    dof = 64 ** 3 * 125 * 5
    for mixed, name in ((True, "mixed"), (False, "fp64")):
        for i, kernel in enumerate(("grad", "rhs")):
            assert bench.profiled_traffic(kernel, name, 4, 64) >= bench.launch_bytes(dof, mixed)[i]
