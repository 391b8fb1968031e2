"""bench.py's command line on the CPU: the multi-GPU request is refused with
a message, tree splits parse as F forests on S streams, and what is reported
of the integrator's launch is what the kernel has."""
import os
import re
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)


def test_more_than_one_gpu_is_refused():
    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"], capture_output=True,
                       text=True, timeout=120)
    assert r.returncode == 2
    assert "measures one GPU" in r.stderr and r.stdout == ""


def test_tree_splits():
    import bench
    assert bench.parse_tree_splits("4,8") == ((4, 4), (8, 8))
    assert bench.parse_tree_splits("4x2, 1, 2") == ((4, 2), (2, 2))
    assert bench.parse_tree_splits("") == ()
    with pytest.raises(ValueError):
        bench.parse_tree_splits("4x0")


def test_reported_launch_is_the_kernel_s():
    import bench
    source = open(os.path.join(ROOT, "galacticus_amd", "csrc", "group_rhs.hpp"), encoding="utf-8").read()
    nodes = int(re.search(r"kGroupNodes = (\d+);", source).group(1))
    waves = int(re.search(r"kGroupWaves = (\d+)", source).group(1))
    assert bench.KERNEL_LAUNCH == {"nodes_per_workgroup": nodes, "workgroups_per_cu": 1, "rhs_waves": waves}


def test_traffic_is_reported_for_the_standard_batch():
    """Whatever shape is set on a handle: one figure for the one kernel."""
    import bench
    assert bench.hbm_traffic(100000, 0) == bench.HBM_TRAFFIC_1E5 > 0.0
    assert bench.hbm_traffic(100000, 1) is None and bench.hbm_traffic(99999, 0) is None
