"""The library's host code without a GPU: allocations that fail, what it
launches and with which arguments.  The HIP runtime is tests/cpp/hip_host.cpp
(host memory, kernels do not run); each case is a function of
tests/host_cases.py in a process of its own."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CASES = ["moved_nodes_of_a_failed_frame", "redwood_stays_inside_wide_images", "bin_capacity_follows_the_factor",
         "closed_objects_free_their_memory", "wide_bins_give_way_to_memory", "readback_by_destination",
         "more_moved_nodes_every_frame", "input_blocks_are_waited_for"]


@pytest.fixture(scope="module", autouse=True)
def runtime():
    # the build step compiles it; a stale or missing library is rebuilt here
    subprocess.run(["make", "-s", "-C", os.path.join(HERE, "cpp")], check=True)


@pytest.mark.parametrize("case", CASES)
def test_case(case):
    out = subprocess.run([sys.executable, os.path.join(HERE, "host_cases.py"), case], capture_output=True, text=True,
                         timeout=120)
    assert out.returncode == 0 and f"case passed: {case}" in out.stdout, out.stdout + out.stderr
