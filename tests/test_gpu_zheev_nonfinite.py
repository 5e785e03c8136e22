"""GPU: zheev of a matrix with a NaN or an infinity reports it (its eigenvalues were whatever
the workspace held), and the next call is not touched by it."""
import numpy as np
import pytest

from test_gpu_parity import ctx  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu

WTB_ERR_NONFINITE = 10


@pytest.mark.parametrize("vectors", [False, True])
@pytest.mark.parametrize("n", [1, 20, 300])
@pytest.mark.parametrize("value", [np.nan, np.inf, 1j * np.inf])
def test_nonfinite_matrix_is_refused(ctx, value, n, vectors):  # noqa: F811
    from wantibexos_amd import bse
    print(f"zheev {value} {n} {vectors}", flush=True)
    rng = np.random.default_rng(n)
    a = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    a = a + a.conj().T
    bad = a.copy()
    bad[0, n - 1] = value if n > 1 else np.real(value) + np.nan
    with pytest.raises(bse.WTBError) as e:
        bse.zheev(ctx, bad, vectors=vectors)
    assert e.value.code == WTB_ERR_NONFINITE
    w = bse.zheev(ctx, a, vectors=vectors)
    w = w[0] if vectors else w
    assert np.linalg.norm(w - np.linalg.eigvalsh(a)) <= 8 * n * np.finfo(float).eps * np.linalg.norm(a)


def test_below_the_diagonal_nothing_is_read(ctx):  # noqa: F811
    from wantibexos_amd import bse
    a = np.diag(np.arange(1.0, 41.0)).astype(complex)
    a[30, 3] = np.nan
    assert np.abs(bse.zheev(ctx, a) - np.arange(1.0, 41.0)).max() < 1e-13
