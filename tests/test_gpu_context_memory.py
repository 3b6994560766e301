"""Device memory of a context that only assembles.

The element-to-nonzero map (4 bytes an entry of every element matrix) is read
by the multigrid's block inversions alone: a context holds it once it is a
level of a hierarchy.  Bars: what a context holds otherwise, computed from the
mesh (MSR columns 4 bytes a nonzero; 28 bytes a coupled node pair, of which
each has at least 9 nonzeros; 4 bytes an element's node pair; 64 bytes an
unknown), plus half of the map.

The first assembly adds the element matrices and residuals, and the continuity
x temperature entries with pressure stabilisation alone; an allocation rounds
up to 2 MB.
"""
import dataclasses

import pytest

from goma_amd import problems

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def test_no_map_without_a_hierarchy():
    from goma_amd import capi

    capi.Context(problems.lid_cavity(n=2, dim=3)).close()  # the library's own first allocations
    free = _free()
    ctx = capi.Context(problems.lid_cavity(n=12, Re=100.0, dim=3, energy=True, Ra=1e3))
    held = free - _free()
    elems = 12 ** 3
    entries = 16 * 27 * 27 + 2 * 3 * 27 * 4 + 16
    print(f"[case] context memory {held / 1e6:.1f} MB, map {4e-6 * elems * entries:.1f} MB", flush=True)
    rest = 4 * ctx.nval + 28 * ctx.nval // 9 + 4 * 27 * 27 * elems + 64 * ctx.N
    assert held <= rest + 2 * elems * entries
    free = _free()
    ctx.attach_multigrid(3)
    assert free - _free() >= 4 * elems * entries
    ctx.close()


@pytest.mark.parametrize("pspg", [0, 1])
def test_assembly_buffers(pspg):
    from goma_amd import capi

    def assemble(n):
        """Bytes of the card that a context's first assembly takes."""
        p = problems.natural_convection(n=n, Ra=1e4)
        ctx = capi.Context(dataclasses.replace(p, phys=dataclasses.replace(p.phys, pspg=pspg, ps_scaling=0.1 * pspg)))
        x, r = (torch.zeros(ctx.N, dtype=torch.float64, device="cuda") for _ in range(2))
        v = torch.zeros(ctx.nval, dtype=torch.float64, device="cuda")
        x += 0.1
        free = _free()
        assert ctx.fill_dev(x.data_ptr(), r.data_ptr(), v.data_ptr()) == 0
        held = free - _free()
        ctx.close()
        return held

    assemble(4)  # the kernels' own code is loaded by their first launch
    n = 256
    held = assemble(n)
    elems = n * n
    kel = 8 * elems * (9 * 81 + 2 * 2 * 9 * 3 + 9)
    re, ct = 8 * elems * 30, 8 * elems * 27
    print(f"[case] assembly memory {held / 1e6:.1f} MB, pspg={pspg}", flush=True)
    want = kel + re + pspg * ct
    assert want <= held <= want + (2 + pspg) * (2 << 20)
