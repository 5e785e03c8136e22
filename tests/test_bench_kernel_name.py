"""CPU: the kernel that the benchmark names beside its times is the one the library's dispatch
runs (plan_default_band and stage1 in csrc)."""
import sys
from pathlib import Path

import pytest

sys.path.insert(0, str(Path(__file__).resolve().parents[1]))


@pytest.mark.parametrize("precision,reduction,band,N,kernel", [
    ("fp64", "auto", 32, 5184, "k_update_mul"), ("fp64", "auto", 32, 16400, "k_update_mul"),
    ("fp64", "auto", 32, 16404, "k_her2k_full"), ("fp64", "auto", 32, 36864, "k_her2k_full"),
    ("fp64", "auto", 16, 36864, "k_her2k_full"), ("fp64", "two", 16, 5184, "k_update_mul"),
    ("fp64", "two", 16, 36864, "k_her2k_full"), ("fp64", "two", 32, 5184, "k_her2k_full"),
    ("mixed", "auto", 32, 14400, "k_her2k_full"), ("mixed", "two", 16, 5184, "k_her2k_full")])
def test_update_kernel(precision, reduction, band, N, kernel):
    import bench
    assert bench.update_kernel(precision, reduction, band, N) == kernel
