"""bench.py's roofline entries on the CPU, from given kernel timings.

The block inversions' flops are those of a launch.
"""
import importlib.util
import os

import pytest

from goma_amd import problems

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def bench():
    spec = importlib.util.spec_from_file_location("bench_roofline", os.path.join(ROOT, "bench.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


def test_block_inversions_flops_are_a_launchs(bench):
    prob = problems.lid_cavity(n=2, Re=100.0, dim=3, energy=True, Ra=1e3)
    n = 27 * 4 + 4
    k = dict(launches=50, total_ms=250.0, avg_ms=5.0, bytes_per_launch=8 * n * n * 20.0, GBps=1.0)
    r = bench.kernel_roofline("k_vanka_invert", k, prob, 0, "none")
    assert r["flops_per_launch"] == 8 * 2 * n ** 3 and "flops_per_assembly" not in r
