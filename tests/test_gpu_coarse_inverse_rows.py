"""The coarsest inverse's rounding, and its row counts around the switches.

Panels of 16 columns with one row a thread up to 256 unknowns, three rows and
256 threads up to 768, three rows and 512 threads up to 1536, panels of 8 and
four rows beyond: 210 / 291, 615 / 770, 1326 / 1623 unknowns, bars of
test_gpu_coarse_inverse.py.

Rounding: a panel's terms of an entry are added up before they reach it.  The
same elimination in NumPy, with partial pivoting and panels of 16, adds the
same terms in other orders, so |G A - I| of the two agree but for chance: within
a quarter in the geometric mean of six states.  (Terms added to the entry one
by one leave 1.6 times as much for 1059 unknowns.)
"""
import numpy as np
import pytest

from goma_amd import problems
from test_gpu_coarse_inverse_edges import _flow, _heat
from test_gpu_coarse_inverse_edges import test_inverse_edges as _check

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

CASES = [("flow-4", lambda: _flow(8), 4, 210), ("flow-8", lambda: _flow(16), 8, 770),
         ("heat-9", lambda: _heat(18), 9, 1326), ("heat-10", lambda: _heat(20), 10, 1623)]


@pytest.mark.parametrize("name,make,nc,ncoarse", CASES, ids=[c[0] for c in CASES])
def test_row_switches(name, make, nc, ncoarse, oracle_mod):
    _check(name, make, nc, ncoarse, oracle_mod)


def _gauss_jordan(A, w=16):
    n, D, perm = len(A), A.copy(), []
    for k0 in range(0, n, w):
        nb = min(w, n - k0)
        P = D[:, k0:k0 + nb].copy()
        swaps = []
        for c in range(nb):
            k = k0 + c
            p = k + int(np.argmax(np.abs(P[k:, c])))
            swaps.append((k, p))
            P[[k, p]] = P[[p, k]]
            inv = 1.0 / P[k, c]
            f = P[:, c] * inv
            row = P[k].copy()
            f[k] = 0.0
            P -= np.outer(f, row)
            P[k] = row * inv
            P[:, c] = -f
            P[k, c] = inv
        rest = np.r_[0:k0, k0 + nb:n]
        for k, p in swaps:
            D[[k, p]] = D[[p, k]]
        B = D[k0:k0 + nb][:, rest].copy()
        D[k0:k0 + nb] = 0.0
        D[:, rest] += P @ B
        D[:, k0:k0 + nb] = P
        perm += swaps
    for k, p in reversed(perm):
        D[:, [k, p]] = D[:, [p, k]]
    return D


def test_rounding(oracle_mod):
    from goma_amd import capi

    ctx = capi.Context(problems.natural_convection(n=16, Ra=1e4, jitter=0.1))
    ctx.attach_multigrid(8)
    cc = ctx._coarse[-1]
    mask, val = ctx.dirichlet()
    ratio = []
    for seed in range(6):
        print(f"[case] coarse inverse rounding N={cc.N} seed={seed}", flush=True)
        x0 = np.random.default_rng(seed).standard_normal(ctx.N) * 0.5
        x0[mask > 0] = val[mask > 0]
        xd = torch.from_numpy(x0).cuda()
        rd, vd, sd = (torch.zeros(k, dtype=torch.float64, device="cuda") for k in (ctx.N, ctx.nval, ctx.N))
        torch.cuda.synchronize()
        assert ctx.fill_dev(xd.data_ptr(), rd.data_ptr(), vd.data_ptr()) == 0
        ctx.row_sum_scale_dev(vd.data_ptr(), rd.data_ptr(), sd.data_ptr())
        ctx.mg_setup_dev(xd.data_ptr(), vd.data_ptr(), sd.data_ptr())
        A = oracle_mod.msr_to_scipy(cc.bindx(), ctx.mg_level_matrix(len(ctx._coarse)), cc.N).toarray()
        eye = np.eye(cc.N)
        ratio.append(np.linalg.norm(ctx.mg_coarse_inverse() @ A - eye) / np.linalg.norm(_gauss_jordan(A) @ A - eye))
    ctx.close()
    assert np.exp(np.mean(np.log(ratio))) <= 1.25, ratio
