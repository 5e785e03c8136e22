"""GPU: the COMPLEX*16 two-stage reduction and its back-transform at the sizes where a tile,
a panel, a row block or a rule of the dispatch ends, against LAPACK.

Tolerances: reduction and back-transform are products of unitary similarities, backward
stable with |dA|_F <= 4 n eps |A|_F (between the sqrt(n) growth that rounding shows and the
n^1.5 of the worst-case bounds).  By Hoffman and Wielandt the eigenvalues of two such solves
differ by at most 8 n eps |A|_F in the 2-norm; the residual and the loss of orthogonality of
the vectors are bounded alike."""
import numpy as np
import pytest

from test_gpu_parity import ctx  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps


def matrix(n, kind):
    rng = np.random.default_rng(n)
    a = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    a = a + a.conj().T
    if kind == "lowrank":                      # columns that are zero below the panel
        a[3:, 3:] = 0.0
    if kind == "banded":                       # reflectors of one element only
        a = np.triu(np.tril(a, 2), -2)
    a[np.diag_indices(n)] = a[np.diag_indices(n)].real
    return a


# 31 | 32: one- and two-stage; 48, 49: panels end; 128 .. 145: row blocks of the update;
# 272 | 273: a panel of one workgroup and of two; 1100: several pieces a wave
@pytest.mark.parametrize("kind", ["dense", "lowrank", "banded"])
@pytest.mark.parametrize("n", [31, 32, 33, 47, 48, 49, 64, 65, 128, 129, 144, 145, 272, 273, 530, 1100])
def test_zheev_edges(ctx, n, kind):
    from wantibexos_amd import bse
    print(f"zheev {n} {kind}", flush=True)
    a = matrix(n, kind)
    norm = np.linalg.norm(a)
    tol = 8 * n * EPS * norm
    ref = np.linalg.eigvalsh(a)
    assert np.linalg.norm(bse.zheev(ctx, np.triu(a)) - ref) <= tol
    w, x = bse.zheev(ctx, np.triu(a), vectors=True)
    assert np.linalg.norm(w - ref) <= tol
    assert np.linalg.norm(a @ x - x * w) <= tol
    assert np.linalg.norm(x.conj().T @ x - np.eye(n)) <= 8 * n * EPS * n ** 0.5


# one row past the sizes where the pass over the trailing matrix takes two and four steps
@pytest.mark.parametrize("n", [3089, 6161])
def test_zheev_invariants(ctx, n):
    from wantibexos_amd import bse
    print(f"zheev {n}", flush=True)
    a = matrix(n, "dense")
    norm = np.linalg.norm(a)
    w = bse.zheev(ctx, np.triu(a))
    assert np.all(np.diff(w) >= 0)
    assert abs(w.sum() - np.trace(a).real) <= n ** 0.5 * 4 * n * EPS * norm
    assert abs((w * w).sum() - norm * norm) <= 2 * norm * 4 * n * EPS * norm
