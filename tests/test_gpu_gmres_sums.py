"""GMRES's projections at the edges of their tiles.

The dot products take eight vectors a block and a power of two of threads a
sum: Krylov spaces of 1 to 120 vectors on both sides of 2, 4, 8, 16, 64, and
vectors from fewer entries than a block to several blocks.  Random matrices,
on which GMRES converges slowly, so that the residual after k iterations is
far from rounding: it must equal the minimum over the Krylov space (Arnoldi
with a second pass, in NumPy) within 1e-9, and the solution's own residual too.
"""
import numpy as np
import pytest

from goma_amd import problems

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _minimum(A, b, k):
    Q, H = [b / np.linalg.norm(b)], np.zeros((k + 1, k))
    for j in range(k):
        w = A @ Q[j]
        for _ in range(2):
            h = np.array([q @ w for q in Q])
            w = w - np.array(Q).T @ h
            H[: j + 1, j] += h
        H[j + 1, j] = np.linalg.norm(w)
        Q.append(w / H[j + 1, j])
    e = np.zeros(k + 1)
    e[0] = 1.0
    y = np.linalg.lstsq(H, e, rcond=None)[0]
    return np.linalg.norm(H @ y - e)


@pytest.mark.parametrize("n,ks", [(3, (1, 2, 3, 4, 7, 8, 9, 31)), (24, (1, 3, 15, 16, 17, 63, 64, 119, 120))])
def test_residual_is_the_minimum(n, ks, oracle_mod):
    from goma_amd import capi

    ctx = capi.Context(problems.lid_cavity(n=n, Re=100.0))
    rng = np.random.default_rng(n)
    val, b = rng.standard_normal(ctx.nval), rng.standard_normal(ctx.N)
    A = oracle_mod.msr_to_scipy(ctx.bindx(), val, ctx.N).tocsr()
    vd, bd = torch.from_numpy(val).cuda(), torch.from_numpy(b).cuda()
    for k in ks:
        print(f"[case] gmres sums n={n} k={k} N={ctx.N}", flush=True)
        xd = torch.zeros(ctx.N, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        its, rel = ctx.gmres_dev(vd.data_ptr(), bd.data_ptr(), xd.data_ptr(), precond=0, kspace=k,
                                 max_its=k, lin_tol=1e-14)
        want = _minimum(A, b, k)
        assert its == k and want > 1e-3
        own = np.linalg.norm(b - A @ xd.cpu().numpy()) / np.linalg.norm(b)
        assert abs(rel - want) <= 1e-9 * want and abs(own - want) <= 1e-9 * want
    ctx.close()


# more blocks of the update than threads that add up its norms (433), and the
# most blocks there are (1024 for 282,882 unknowns)
@pytest.mark.parametrize("n", [100, 160])
def test_many_blocks(n, oracle_mod):
    test_residual_is_the_minimum(n, (2, 9), oracle_mod)
