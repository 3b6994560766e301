"""The ILU(0) sweeps on Jacobians, and on pivots out of the normal range.

One GMRES iteration from a zero guess returns a multiple z of M^-1 b.  Solving
L U z = alpha b by substitution leaves at most 2 (n + 2) eps |L| |U| |z| a row,
n the longest row, whatever the nodes' triangles (saddle points make them
ill-conditioned); the bar is that in the 2-norm, twice over for alpha's own
rounding.  States are those where products with the triangles' inverses leave
up to 100 times the bar.

A decoupled unknown with a pivot whose reciprocal overflows, or is subnormal,
is still divided by it: every decoupled unknown must give the same alpha, to
the 1e-10 that subnormal inputs keep.
"""
import numpy as np
import pytest
import scipy.sparse as sp

from goma_amd import problems

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _apply(ctx, val, b, bins):
    vd, bd = torch.from_numpy(val).cuda(), torch.from_numpy(b).cuda()
    xd = torch.zeros(ctx.N, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    ctx.gmres_dev(vd.data_ptr(), bd.data_ptr(), xd.data_ptr(), kspace=1, max_its=1, lin_tol=1e-30, precond=1,
                  patch_bins=bins)
    return vd, xd.cpu().numpy()


CASES = [("carreau2d", s, lambda s: problems.natural_convection(n=8, Ra=1e4, carreau=True, jitter=0.15, seed=s))
         for s in range(4)]
CASES += [("cavity3d", s, lambda s: problems.lid_cavity(n=3, Re=400.0, dim=3, energy=True, Ra=1e4)) for s in range(8)]


@pytest.mark.parametrize("name,seed,make", CASES, ids=[f"{c[0]}-{c[1]}" for c in CASES])
def test_sweeps_are_substitution(name, seed, make, oracle_mod):
    from goma_amd import capi

    prob = make(seed)
    print(f"[case] ilu substitution {name} seed={seed}", flush=True)
    ctx = capi.Context(prob)
    orc = oracle_mod.Oracle(prob)
    rc, r, v = orc.fill(np.random.default_rng(seed).standard_normal(orc.N) * 0.3)
    s = np.zeros(orc.N)
    oracle_mod.lib().om_row_sum_scale(orc.N, v, orc.ija, r, s)
    vd, z = _apply(ctx, v, r, 2)
    rowptr, col, lu = ctx.ilu0_factor_dev(vd.data_ptr(), 2)
    perm, _ = ctx.patch_permutation(2)
    ctx.close()
    F = sp.csr_matrix((lu, col, rowptr), shape=(orc.N, orc.N))
    L, U = (sp.tril(F, -1) + sp.identity(orc.N)).tocsr(), sp.triu(F).tocsr()
    z, pb = z[perm], r[perm]
    t = L @ (U @ z)
    alpha = (t @ pb) / (pb @ pb)
    n = np.diff(rowptr).max()
    bar = 4 * (n + 2) * np.finfo(float).eps * np.linalg.norm(abs(L) @ (abs(U) @ abs(z)))
    assert np.linalg.norm(t - alpha * pb) <= bar


@pytest.mark.parametrize("dim,energy", [(2, False), (2, True), (3, True)])
@pytest.mark.parametrize("pivot,rhs", [(1e-310, 1e-311), (1.5 * 2.0 ** 1023, 1e100), (-1e-310, 1e-311)])
def test_pivots_out_of_the_normal_range(dim, energy, pivot, rhs):
    from goma_amd import capi

    if dim == 2:
        prob = problems.natural_convection(n=3, Ra=1e3) if energy else problems.lid_cavity(n=3)
    else:
        prob = problems.lid_cavity(n=2, Re=100.0, dim=3, energy=True, Ra=1e3)
    ctx = capi.Context(prob)
    N = ctx.N
    bindx = ctx.bindx()
    print(f"[case] ilu pivot {pivot} dim={dim} energy={energy} N={N}", flush=True)
    rng = np.random.default_rng(3)
    val = np.zeros(ctx.nval)
    val[:N] = 2.0
    b = rng.uniform(1.0, 2.0, N)
    odd = np.arange(0, N, 7)
    val[odd] = pivot
    b[odd] = rhs
    _, z = _apply(ctx, val, b, 1)
    ctx.close()
    alpha = z * val[:N] / b
    ref = np.median(alpha[np.setdiff1d(np.arange(N), odd)])
    assert np.isfinite(z).all() and ref != 0.0
    assert np.abs(alpha / ref - 1.0).max() <= 1e-10
