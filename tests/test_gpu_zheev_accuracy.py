"""GPU: the residual of zheev's eigenvectors.  The reduction rounds an element once a panel of
32 columns, and so does the back-transform, n / 32 panels each; with the divide and conquer
three such sums of random half units, (n / 32)^1/2 / 2 each, so |A X - X W|_F stays below
2 (n / 32)^1/2 eps |A|_F.  A reduction that takes every row through n more transformations
does not."""
import numpy as np
import pytest

from test_gpu_parity import ctx  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [640, 1001, 1290])
def test_vectors_residual(ctx, n):  # noqa: F811
    from wantibexos_amd import bse
    rng = np.random.default_rng(n)
    a = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    a = (a + a.conj().T) / n ** 0.5
    a[np.diag_indices(n)] = rng.uniform(2.0, 10.0, n)
    w, x = bse.zheev(ctx, np.triu(a), vectors=True)
    eps = np.finfo(float).eps
    res = np.linalg.norm(a @ x - x * w) / np.linalg.norm(a) / eps
    print(f"n {n}: residual {res:.1f} eps", flush=True)
    assert res <= 2 * (n / 32) ** 0.5
    assert np.linalg.norm(x.conj().T @ x - np.eye(n)) <= 2 * (n / 32) ** 0.5 * eps * n ** 0.5 * 2
