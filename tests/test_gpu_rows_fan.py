"""The HEX27 row kernel on a node pattern too long for four waves' LDS.

Hexahedra around a common edge: the edge's nodes see every other node, 24
elements give them 1836 columns (rows of ~460 neighbours, read in several
rounds of 64), where the kernel takes two nodes per workgroup instead of
four.  Bar of test_gpu_rows.py: 1e-13 of max|A x|.
"""
from dataclasses import replace

import numpy as np
import pytest

from goma_amd import mesh as M
from goma_amd import problems

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def fan(k):
    """k hexahedra around the z axis, each with the quadrilateral (axis, p_i, m_i, p_i+1)."""
    loc = M.structured_mesh(3, 1)
    ref = loc.coor[:, loc.connect[0]].T  # the element's nodes in [0, 1]^3, local order
    xy = lambda r, t: np.array([r * np.cos(2 * np.pi * t / k), r * np.sin(2 * np.pi * t / k)])
    nodes, ids, conn = [], {}, np.empty((k, 27), np.int32)
    for e in range(k):
        q = [np.zeros(2), xy(1.0, e), xy(1.3, e + 0.5), xy(1.0, (e + 1) % k)]
        for i, (s, t, u) in enumerate(ref):
            p = (1 - s) * (1 - t) * q[0] + s * (1 - t) * q[1] + s * t * q[2] + (1 - s) * t * q[3]
            key = (round(p[0] * 1e6), round(p[1] * 1e6), round(u * 1e6))
            if key not in ids:
                ids[key] = len(nodes)
                nodes.append((p[0], p[1], u))
            conn[e, i] = ids[key]
    return M.Mesh(dim=3, n=0, coor=np.ascontiguousarray(np.array(nodes).T), connect=conn)


@pytest.mark.parametrize("k,cap", [(24, 1836), (20, 1532)])
def test_matvec_on_a_fan(k, cap, oracle_mod):
    from goma_amd import capi

    base = problems.lid_cavity(n=1, Re=100.0, dim=3, energy=True, Ra=1e3)
    mesh = fan(k)
    prob = replace(base, mesh=mesh, dbc_node=base.dbc_node[:0], dbc_var=base.dbc_var[:0],
                   dbc_value=base.dbc_value[:0])
    assert mesh.num_nodes == 18 * k + 3 and 4 * mesh.num_nodes + 4 * k == cap
    ctx = capi.Context(prob)
    print(f"[case] fan of {k} N={ctx.N}", flush=True)
    rng = np.random.default_rng(5)
    val, x = rng.standard_normal(ctx.nval), rng.standard_normal(ctx.N)
    A = oracle_mod.msr_to_scipy(ctx.bindx(), val, ctx.N)
    assert np.diff(A.tocsr().indptr).max() == cap
    vd, xd = torch.from_numpy(val).cuda(), torch.from_numpy(x).cuda()
    yd = torch.zeros(ctx.N, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    ctx.matvec_dev(vd.data_ptr(), xd.data_ptr(), yd.data_ptr())
    torch.cuda.synchronize()
    ref = A @ x
    assert np.abs(yd.cpu().numpy() - ref).max() <= 1e-13 * np.abs(ref).max()
    ctx.close()
