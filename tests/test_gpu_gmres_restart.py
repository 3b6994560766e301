"""GMRES restart lengths past the stand-alone solver's 120, through Newton.

One Newton pass whose linear solve is a single unpreconditioned cycle of k
vectors, on both sides of 128 (a thread per projection from 129 sums on) and
256 (more sums than threads).  The Krylov spaces are nested, so the residual
falls with k; it is the returned correction's own residual (in the pass's own
matrix, to 64 eps |A| |dx|); and 300 vectors reduce it below 1e-9, as they do
in exact arithmetic (4e-11 in NumPy), where any projection lost or misread
from the 128th on leaves it near the 1e-3 of 127 vectors.  Lengths that no
cycle could use are refused before anything runs, the state untouched.
"""
import numpy as np
import pytest

from goma_amd import problems

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

LENGTHS = (127, 128, 129, 200, 255, 256, 257, 300)


@pytest.fixture(scope="module")
def cavity():
    from goma_amd import capi

    ctx = capi.Context(problems.lid_cavity(n=7, Re=100.0))
    x0 = np.random.default_rng(1).standard_normal(ctx.N) * 0.3
    yield capi, ctx, x0
    ctx.close()


def test_long_cycles(cavity, oracle_mod):
    capi, ctx, x0 = cavity
    xd = torch.from_numpy(x0).cuda()
    r, v, s = (torch.zeros(k, dtype=torch.float64, device="cuda") for k in (ctx.N, ctx.nval, ctx.N))
    torch.cuda.synchronize()
    assert ctx.fill_dev(xd.data_ptr(), r.data_ptr(), v.data_ptr()) == 0
    ctx.row_sum_scale_dev(v.data_ptr(), r.data_ptr(), s.data_ptr())
    A = oracle_mod.msr_to_scipy(ctx.bindx(), v.cpu().numpy(), ctx.N).tocsr()
    b = r.cpu().numpy()
    last = 1.0
    for k in LENGTHS:
        print(f"[case] gmres restart length {k} N={ctx.N}", flush=True)
        xd = torch.from_numpy(x0).cuda()
        torch.cuda.synchronize()
        _, rep = ctx.solve_dev(xd.data_ptr(), precond=0, kspace=k, max_its=k, lin_tol=1e-15, max_newton=1)
        assert rep.lin_its[0] == k
        dx = x0 - xd.cpu().numpy()
        own = np.linalg.norm(b - A @ dx) / np.linalg.norm(b)
        slack = 64 * np.finfo(float).eps * np.linalg.norm(abs(A) @ abs(dx) + abs(A) @ abs(x0)) / np.linalg.norm(b)
        assert abs(rep.lin_relres[0] - own) <= slack, (k, rep.lin_relres[0], own, slack)
        assert rep.lin_relres[0] < last, k
        last = rep.lin_relres[0]
    assert last <= 1e-9


@pytest.mark.parametrize("kspace,max_its", [(0, 10), (-3, 10), (4095, 4095)])
def test_lengths_out_of_range_are_refused(cavity, kspace, max_its):
    capi, ctx, x0 = cavity
    print(f"[case] gmres restart length {kspace} refused", flush=True)
    xd = torch.from_numpy(x0).cuda()
    torch.cuda.synchronize()
    with pytest.raises(RuntimeError, match="restart length"):
        ctx.solve_dev(xd.data_ptr(), precond=0, kspace=kspace, max_its=max_its, max_newton=1)
    assert np.array_equal(xd.cpu().numpy(), x0)


def test_a_length_beyond_the_iteration_limit_is_taken(cavity):
    capi, ctx, x0 = cavity
    print("[case] gmres restart length 4095, 5 iterations", flush=True)
    out = []
    for k in (5, 4095):
        xd = torch.from_numpy(x0).cuda()
        torch.cuda.synchronize()
        _, rep = ctx.solve_dev(xd.data_ptr(), precond=0, kspace=k, max_its=5, lin_tol=1e-15, max_newton=1)
        assert rep.lin_its[0] == 5
        out.append(xd.cpu().numpy())
    assert np.array_equal(out[0], out[1])


def test_longest_cycle():
    from goma_amd import capi

    ctx = capi.Context(problems.lid_cavity(n=22, Re=100.0))
    print(f"[case] gmres restart length 4094 N={ctx.N}", flush=True)
    xd = torch.from_numpy(np.random.default_rng(1).standard_normal(ctx.N) * 0.3).cuda()
    torch.cuda.synchronize()
    _, rep = ctx.solve_dev(xd.data_ptr(), precond=0, kspace=4094, max_its=4094, lin_tol=1e-30, max_newton=1)
    assert rep.lin_its[0] == 4094 and rep.lin_relres[0] <= 1e-9
    ctx.close()
