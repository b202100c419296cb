"""bench.py: which measured traffic it prints beside the deposit's times."""
import json
import os
import re
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
import bench  # noqa: E402


@pytest.mark.parametrize("kernel,taken", [
    ("void k_gather_full<2752, false> + void k_gather_full<448, true> + void k_gather_light<true>", True),
    ("void k_gather_march<2752, false> + void k_gather_slab<2752, false> + void k_gather_light<true>", False),
    ("void k_gather_light<true>", False)])
def test_traffic_is_of_the_timed_kernels(tmp_path, kernel, taken):
    path = str(tmp_path / "t.json")
    with open(path, "w") as f:
        json.dump({"kernel": kernel, "workload": "cfg1_0_1001", "bytes_per_launch": 1.0, "source": "s"}, f)
    assert (bench.load_traffic("cfg1_0_1001", path) is not None) == taken
    assert bench.load_traffic("cfg3_0_1003", path) is None


def test_timed_kernels_exist():
    with open(os.path.join(ROOT, "ahf_amd", "csrc", "amr_gpu.hip")) as f:
        src = f.read()
    for k in bench.DEPOSIT_KERNELS:
        assert re.search(r"__global__[^;{]*\b%s\(" % k, src), k
