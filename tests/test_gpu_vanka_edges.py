"""QUAD9 element-block inverses in part-filled workgroups, with and without energy.

Eight blocks share a workgroup, two a wave: 36 and 100 elements leave four in
the last.  Blocks of 21 and of 30 unknowns.  The checks and bars of
test_gpu_vanka.py (whose cases are 16 elements with energy).
"""
import pytest

import test_gpu_vanka as V
from goma_amd import problems

pytestmark = pytest.mark.gpu

CASES = {
    "quad9_ns_36": lambda: problems.lid_cavity(n=6, Re=100.0, jitter=0.1),
    "quad9_energy_100": lambda: problems.natural_convection(n=10, Ra=1e4, jitter=0.1),
    "quad9_carreau_36": lambda: problems.natural_convection(n=6, Ra=1e4, carreau=True, jitter=0.1),
}


@pytest.mark.parametrize("name", list(CASES))
def test_block_inverses_of_partial_workgroups(name, monkeypatch, oracle_mod):
    from goma_amd import capi

    monkeypatch.setitem(V.CASES, name, CASES[name])
    V.test_block_inverses_match_lapack(name, capi, oracle_mod)
