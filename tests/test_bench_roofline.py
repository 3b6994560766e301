"""bench.py's roofline entries on the CPU, from given kernel timings.

The assembly's fraction of peak counts the bytes that the call cannot do
without; the element matrices that its kernels write and read again do not
raise it.  The block inversions' flops are those of a launch.
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


@pytest.mark.parametrize("scratch", [0.0, 24e9])
def test_assembly_fraction_counts_the_calls_bytes(bench, scratch):
    prob = problems.lid_cavity(n=2, Re=100.0, dim=3, energy=True, Ra=1e3)
    # 11 assemblies of two launches, 10 ms each, 8 GB compulsory
    k = dict(launches=22, total_ms=110.0, avg_ms=5.0, bytes_per_launch=(8e9 + scratch) / 2)
    r = bench.assembly_roofline(k, 11, 8e9, prob, "none")
    assert r["per_assembly_s"] == 0.01 and r["achieved"] == 800.0 and r["frac"] == 0.1
    assert r["bytes_per_assembly"] == 8e9 and r["kernel_bytes_per_assembly"] == 8e9 + scratch
    # 8 elements, 4 waves of 7 (5 + 3 * 6 + 3) + 14 products of 2048 flop
    assert r["mfma"]["flops_per_assembly"] == 8 * 4 * (7 * 26 + 14) * 2048


def test_block_inversions_flops_are_a_launchs(bench):
    prob = problems.lid_cavity(n=2, Re=100.0, dim=3, energy=True, Ra=1e3)
    n = 27 * 4 + 4
    k = dict(launches=50, total_ms=250.0, avg_ms=5.0, bytes_per_launch=8 * n * n * 20.0, GBps=1.0)
    r = bench.kernel_roofline("k_vanka_invert", k, prob, 0, "none")
    assert r["flops_per_launch"] == 8 * 2 * n ** 3 and "flops_per_assembly" not in r
