"""A band that does not fit the card: refused, with nothing kept.

A shuffled 140 x 140 mesh has 216,000 unknowns and a band as wide as the
matrix, 750 GB.  The refused factorisation leaves the card's free memory as it
was (to 2 MB, an allocation's granularity; the inverse triangles and solve
operators of these unknowns are 660 MB), a second call is refused the same way,
and the context still solves without the preconditioner.
"""
import dataclasses

import numpy as np
import pytest

from goma_amd import problems
from goma_amd.mesh import renumber

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def test_refused_band_keeps_nothing():
    from goma_amd import capi

    p = problems.lid_cavity(n=140)
    rng = np.random.default_rng(5)
    order = rng.permutation(p.mesh.num_nodes)
    new = np.empty_like(order)
    new[order] = np.arange(order.size)
    mesh = renumber(p.mesh, order, rng.permutation(p.mesh.num_elems))
    ctx = capi.Context(dataclasses.replace(p, mesh=mesh, dbc_node=new[p.dbc_node].astype(np.int32)))
    print(f"[case] refused band N={ctx.N}", flush=True)
    val = np.zeros(ctx.nval)
    val[: ctx.N] = 2.0
    b = rng.standard_normal(ctx.N)
    vd, bd = torch.from_numpy(val).cuda(), torch.from_numpy(b).cuda()
    xd = torch.zeros(ctx.N, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()

    def solve(precond):
        return ctx.gmres_dev(vd.data_ptr(), bd.data_ptr(), xd.data_ptr(), kspace=2, max_its=2, lin_tol=1e-12,
                             precond=precond)

    solve(0)
    free = torch.cuda.mem_get_info()[0]
    for _ in range(2):
        with pytest.raises(RuntimeError, match="banded LU needs"):
            solve(3)
        assert torch.cuda.mem_get_info()[0] >= free - (2 << 20)
    xd.zero_()
    torch.cuda.synchronize()
    solve(0)
    assert np.abs(xd.cpu().numpy() - b / 2.0).max() <= 1e-12 * np.abs(b).max()
    ctx.close()
