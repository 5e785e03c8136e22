"""GPU: the two-stage reduction's tracked vectors, its kept reflectors and the sizes where its
form changes, against the one-stage reduction of the same matrix.

Energies: both reductions are backward stable with |dA|_F <= 4 n eps |A|_F, so by Hoffman and
Wielandt the energies differ by at most 8 n eps |W| in the 2-norm.  eps(omega) at width
s >= 0.05 eV is a Lipschitz function of the matrix (|d(H - z)^-1| <= |dA| / s^2); 1e-9 of its
largest value leaves that a factor of a thousand at these sizes."""
import numpy as np
import pytest

from test_gpu_parity import ctx  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps


def model():
    from wantibexos_amd import tbmodel
    return tbmodel.hex2d(seed=9, nw=6, ngrid=(12, 12, 1))


def params(n1, n2, **kw):
    from wantibexos_amd import bse
    return bse.BSEParams(ngrid=(n1, n2, 1), nc=2, nv=2, coultype="V2DRK", r0=40.0, cshift=0.05, ebse0=0.0,
                         ebsef=6.0, numbse=201, dtfull=True, cpol=True, f154=False, **kw)


def run(ctx, prm, *reduction):
    from wantibexos_amd import bse
    with bse.BSEPlan(ctx, model(), prm) as plan:
        if reduction:
            plan.set_reduction(*reduction)
        plan.execute()
        return plan.results()


def compare(got, ref):
    n = len(ref["W"])
    assert np.linalg.norm(got["W"] - ref["W"]) <= 8 * n * EPS * np.linalg.norm(ref["W"])
    assert np.abs(got["eps"] - ref["eps"]).max() <= 1e-9 * np.abs(ref["eps"]).max()
    scale = np.abs(ref["act"]).max()
    assert np.abs(got["act"].sum(axis=1) - ref["act"].sum(axis=1)).max() <= 1e-10 * n * scale


# one and two panels and their ends, row blocks of 128, one and two workgroups a panel, several
@pytest.mark.parametrize("grid", [(2, 4), (3, 3), (3, 4), (1, 13), (4, 4), (4, 8), (3, 11), (4, 9), (4, 17), (3, 23),
                                  (11, 12), (1, 257)])
@pytest.mark.parametrize("temp", [0.0, 3000.0])
def test_tracked_vectors(ctx, grid, temp):  # noqa: F811
    print(f"tracked {grid} T {temp}", flush=True)
    prm = params(*grid, **(dict(bset=True, temp=temp, ta="VE", st=0.3, phavg=0.05) if temp else {}))
    compare(run(ctx, prm), run(ctx, prm, False))


# 16400: the last size of one-launch panels (64 workgroups, band 16); above: band 32
@pytest.mark.parametrize("grid", [(50, 82), (54, 76)])
def test_largest_one_launch_panel(ctx, grid):  # noqa: F811
    print(f"grid {grid}, N = {4 * grid[0] * grid[1]}", flush=True)
    prm = params(*grid)
    compare(run(ctx, prm), run(ctx, prm, False))


# the iterative solver's small solves: the first basis of nev + guard vectors, then up to
# max_sub; the coarse block (3001: past N m = 3000^2, one-stage).  A context whose waits give up
# at once takes the one-stage form for all of them.  Without a coarse block of some size the
# solver does not reach 1e-8 in its 60 iterations, in either form.
@pytest.mark.parametrize("nev,guard,max_sub,coarse,tol", [
    (16, 15, 64, 0, 1e-6), (16, 16, 64, 33, 1e-6), (20, 27, 200, 145, 1e-8), (33, 32, 300, 273, 1e-8),
    (64, 66, 520, 1100, 1e-8), (16, 16, 200, 3001, 1e-8)])
def test_small_solves(ctx, nev, guard, max_sub, coarse, tol):  # noqa: F811
    from wantibexos_amd import bse
    print(f"lowest nev {nev} guard {guard} sub {max_sub} coarse {coarse}", flush=True)
    prm = params(28, 28, precision=bse.MIXED)

    def lowest(c):
        with bse.BSEPlan(c, model(), prm) as plan:
            return plan.lowest(nev=nev, guard=guard, max_sub=max_sub, coarse=coarse, tol=tol, lanczos_steps=0,
                               fallback=False, vectors=True)
    got = lowest(ctx)
    with bse.Context(0) as hasty:
        hasty.set_wait_limit(1)
        ref = lowest(hasty)
    assert got["resid"].max() <= tol
    assert np.abs(got["W"] - ref["W"]).max() <= 2 * tol      # either within its residual of an energy
    x = got["X"]
    assert np.linalg.norm(x.conj().T @ x - np.eye(nev)) < 1e-10
    if coarse >= 145:
        # the block preconditions: a wrong one would cost iterations
        assert abs(got["info"]["iters"] - ref["info"]["iters"]) <= 1
