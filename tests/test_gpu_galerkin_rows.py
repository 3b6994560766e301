"""Galerkin coarse operators without the energy equation, and in FP32.

Each block row of a coarse element is a workgroup of its own (HEX27) or one for
all (QUAD9), with two to four columns per node pair: the forms that
test_gpu_galerkin.py does not reach, against the same R A P.  Bars: 1e-12 of
the largest entry in FP64, 1e-6 in FP32.
"""
import numpy as np
import pytest

from goma_amd import problems
from test_gpu_galerkin import _natural

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

CASES = {
    "cavity2d": lambda: problems.lid_cavity(n=8, Re=100.0, jitter=0.1),
    "natconv2d_odd": lambda: problems.natural_convection(n=6, Ra=1e4, jitter=0.1),
    "cavity3d": lambda: problems.lid_cavity(n=4, Re=100.0, dim=3, jitter=0.1),
    "cavity3d_energy": lambda: problems.lid_cavity(n=4, Re=100.0, dim=3, energy=True, Ra=1e3),
}


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("name", list(CASES))
def test_coarse_rows(name, mixed, oracle_mod):
    import scipy.sparse as sp
    from goma_amd import capi

    prob = CASES[name]()
    print(f"[case] galerkin rows {name} mixed={mixed}", flush=True)
    ctx = capi.Context(prob)
    nl = ctx.attach_multigrid(2)
    assert nl >= 2
    x0 = np.random.default_rng(11).standard_normal(ctx.N) * 0.3
    mask, val = ctx.dirichlet()
    x0[mask > 0] = val[mask > 0]
    xd = torch.from_numpy(x0.copy()).cuda()
    ctx.solve_dev(xd.data_ptr(), max_newton=1, precond=2, mg_galerkin=1, kspace=10, max_its=2,
                  precision=int(mixed))
    orc = oracle_mod.Oracle(_natural(prob))
    rc, _, v = orc.fill(x0)
    assert rc == 0
    A = oracle_mod.msr_to_scipy(orc.ija, v, orc.N)
    rp, ci, cv = ctx.mg_prolongation(1)
    cc = ctx._coarse[0]
    P = sp.csr_matrix((cv, ci, rp), shape=(ctx.N, cc.N))
    A = (P.T @ A @ P).tocsr()
    G = oracle_mod.msr_to_scipy(cc.bindx(), ctx.mg_level_matrix(1), cc.N).tocsr()
    free = np.flatnonzero(cc.dirichlet()[0] == 0)
    err = abs(G[free] - A[free]).max()
    assert err <= (1e-6 if mixed else 1e-12) * abs(A).max(), err
    ctx.close()
