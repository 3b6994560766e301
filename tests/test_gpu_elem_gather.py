"""Element assembly at the edges of its workgroups, and its order.

Four QUAD9 elements share a workgroup (one HEX27) and a thread sums a pair of nodes: one to five
elements leave every remainder of a workgroup, a renumbered mesh every order of
a pair's two nodes (columns before and after the row's own unknown).  Every
form of the kernel (energy or not, constant or shear-thinning viscosity), with
the terms that only some elements have.  Bars: residual and Jacobian within
1e-12 of the oracle's largest entry (FP32 Jacobian 1e-6), stored over a
NaN-filled array and added to a filled one; two assemblies give the same bits.
"""
from dataclasses import replace

import numpy as np
import pytest

from goma_amd import problems
from goma_amd.mesh import renumber

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _cut(prob, ne):
    """The first ne elements of the mesh (a prefix of its rows), renumbered at random."""
    m = prob.mesh
    conn = m.connect[:ne]
    nodes = np.unique(conn)
    new = np.full(m.num_nodes, -1, np.int64)
    new[nodes] = np.arange(nodes.size)
    mesh = replace(m, coor=np.ascontiguousarray(m.coor[:, nodes]),
                   connect=np.ascontiguousarray(new[conn].astype(m.connect.dtype)))
    keep = new[prob.dbc_node] >= 0
    node = new[prob.dbc_node[keep]]
    rng = np.random.default_rng(ne)
    order = rng.permutation(nodes.size)
    inv = np.empty_like(order)
    inv[order] = np.arange(order.size)
    return replace(prob, mesh=renumber(mesh, order, rng.permutation(ne)),
                   dbc_node=inv[node].astype(np.int32), dbc_var=prob.dbc_var[keep],
                   dbc_value=prob.dbc_value[keep])


def _make(kind, ne):
    n = 4 if ne > 4 else ne
    if kind == "flow":
        p = problems.lid_cavity(n=n, Re=100.0, jitter=0.1)
    elif kind == "carreau":
        p = problems.natural_convection(n=n, Ra=1e4, carreau=True, jitter=0.1)
    else:
        p = problems.natural_convection(n=n, Ra=1e4, jitter=0.1)
    if kind == "stabilised":
        p = replace(p, phys=replace(p.phys, pspg=1, ps_scaling=0.5, energy_supg=1.0))
    return _cut(p, ne)


@pytest.mark.parametrize("kind", ["flow", "energy", "carreau", "stabilised"])
@pytest.mark.parametrize("ne", [1, 2, 3, 5])
def test_assembly_at_workgroup_edges(kind, ne, oracle_mod):
    _check(_make(kind, ne), kind, ne, oracle_mod)


@pytest.mark.parametrize("kind", ["flow", "energy", "carreau", "stabilised", "carreau_flow"])
@pytest.mark.parametrize("ne", [1, 3])
def test_hex_assembly(kind, ne, oracle_mod):
    n = 2 if ne > 1 else 1
    if kind in ("flow", "carreau_flow"):
        p = problems.lid_cavity(n=n, Re=100.0, dim=3, jitter=0.1)
        if kind == "carreau_flow":
            q = problems.natural_convection(n=1, Ra=1e4, dim=3, carreau=True).phys
            p = replace(p, phys=replace(q, energy=p.phys.energy))
    elif kind == "carreau":
        p = problems.natural_convection(n=n, Ra=1e4, dim=3, carreau=True, jitter=0.1)
    else:
        p = problems.lid_cavity(n=n, Re=100.0, dim=3, energy=True, Ra=1e3, jitter=0.1)
    if kind == "stabilised":
        p = replace(p, phys=replace(p.phys, pspg=1, ps_scaling=0.5, energy_supg=1.0))
    _check(_cut(p, ne), kind, ne, oracle_mod)


def _check(prob, kind, ne, oracle_mod):
    from goma_amd import capi

    ctx, orc = capi.Context(prob), oracle_mod.Oracle(prob)
    print(f"[case] element gather {kind} ne={ne} N={ctx.N}", flush=True)
    assert prob.mesh.connect.shape[0] == ne
    if kind == "energy":
        e, sd = np.zeros(1, np.int32), np.ones(1, np.int32)
        ctx.add_qconv(e, sd, 1.3, 0.4)
        assert orc.add_qconv(e, sd, 1.3, 0.4) == 0
        ctx.add_qside(e + ne - 1, sd, -0.3)
        assert orc.add_qside(e + ne - 1, sd, -0.3) == 0
    if kind == "stabilised":
        ctx.set_velocity_norm(0.7)
        orc.set_velocity_norm(0.7)
    x = np.random.default_rng(3).standard_normal(ctx.N) * 0.5
    rc, R, V = orc.fill(x)
    assert rc == 0
    xd = torch.from_numpy(x).cuda()

    def run(call, dtype, fill):
        r = torch.zeros(ctx.N, dtype=torch.float64, device="cuda")
        v = torch.full((ctx.nval,), fill, dtype=dtype, device="cuda")
        torch.cuda.synchronize()
        assert call(xd.data_ptr(), r.data_ptr(), v.data_ptr()) == 0
        v = v.cpu().numpy().astype(np.float64)
        v[ctx.N] = V[ctx.N]
        return r.cpu().numpy(), v

    tol = 1e-12 * np.abs(V).max()
    r, v = run(ctx.fill_assign_dev, torch.float64, float("nan"))
    assert np.abs(r - R).max() <= 1e-12 * np.abs(R).max()
    assert np.abs(v - V).max() <= tol
    r2, v2 = run(ctx.fill_assign_dev, torch.float64, -7.0)
    assert np.array_equal(r2, r) and np.array_equal(v2, v)
    _, va = run(ctx.fill_dev, torch.float64, 1.0)
    va[: ctx.N] -= 1.0
    va[ctx.N + 1:] -= 1.0
    assert np.abs(va - V).max() <= tol + 1e-12
    _, v32 = run(ctx.fill32_dev, torch.float32, 0.0)
    assert np.abs(v32 - V).max() <= 1e-6 * np.abs(V).max()
    ctx.close()
