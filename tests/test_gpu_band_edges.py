"""The banded LU at the edges of its panels, tiles and solve steps.

Random diagonally dominant values on the contexts' own graphs (no growth
without pivoting), so one GMRES iteration preconditioned by the FP64 LU leaves
a residual of a few N eps: the bar is 1e-12.  Sizes: N below one panel, one
panel and a few unknowns, N at and around multiples of the 64-column panel and
the 128-unknown solve step, bandwidths from under one panel to many tiles, a
different lower and upper reach, 2D and 3D.
"""
import numpy as np
import pytest

from goma_amd import problems
from goma_amd.mesh import renumber

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _strip(n, keep):
    """The first `keep` rows of elements of an n x n cavity mesh (its own nodes)."""
    import dataclasses

    p = problems.lid_cavity(n=n)
    m = p.mesh
    nodes = (2 * n + 1) * (2 * keep + 1)
    mesh = dataclasses.replace(m, coor=np.ascontiguousarray(m.coor[:, :nodes]),
                               connect=np.ascontiguousarray(m.connect[: n * keep]))
    k = p.dbc_node < nodes
    return dataclasses.replace(p, mesh=mesh, dbc_node=p.dbc_node[k], dbc_var=p.dbc_var[k],
                               dbc_value=p.dbc_value[k])


def _shuffled():
    p = problems.natural_convection(n=5, Ra=1e3)
    rng = np.random.default_rng(2)
    order = rng.permutation(p.mesh.num_nodes)
    new = np.empty_like(order)
    new[order] = np.arange(order.size)
    import dataclasses

    mesh = renumber(p.mesh, order, rng.permutation(p.mesh.num_elems))
    return dataclasses.replace(p, mesh=mesh, dbc_node=new[p.dbc_node].astype(np.int32))


CASES = [("one-element", lambda: problems.lid_cavity(n=1)), ("strip-1x3", lambda: _strip(1, 1)),
         ("strip-3", lambda: _strip(3, 1)), ("n3", lambda: problems.lid_cavity(n=3)),
         ("strip-8x2", lambda: _strip(8, 2)), ("n6-energy", lambda: problems.natural_convection(n=6, Ra=1e3)),
         ("strip-24x2", lambda: _strip(24, 2)), ("n13", lambda: problems.lid_cavity(n=13)),
         ("full-band", _shuffled),
         ("hex-n3", lambda: problems.lid_cavity(n=3, Re=100.0, dim=3, energy=True, Ra=1e3))]


@pytest.mark.parametrize("name,make", CASES, ids=[c[0] for c in CASES])
def test_band_lu_is_a_direct_solve(name, make, oracle_mod):
    from goma_amd import capi

    ctx = capi.Context(make())
    N, bindx = ctx.N, ctx.bindx()
    print(f"[case] band edges {name} N={N}", flush=True)
    rng = np.random.default_rng(11)
    val = rng.uniform(-1.0, 1.0, ctx.nval)
    length = np.diff(bindx[: N + 1])
    val[N + 1:] /= np.repeat(np.maximum(length, 1), length)
    val[:N] = 2.0
    b = rng.standard_normal(N)
    vd, bd = torch.from_numpy(val).cuda(), torch.from_numpy(b).cuda()
    zd = torch.zeros(N, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    its, _ = ctx.gmres_dev(vd.data_ptr(), bd.data_ptr(), zd.data_ptr(), kspace=4, max_its=1,
                           lin_tol=1e-30, precond=3)
    ctx.close()
    A = oracle_mod.msr_to_scipy(bindx, val, N)
    assert its == 1
    assert np.linalg.norm(b - A @ zd.cpu().numpy()) <= 1e-12 * np.linalg.norm(b)
