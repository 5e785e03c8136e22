"""GPU: the bounded waits between the workgroups of the two-stage reduction.  With a limit of
one poll every wait gives up at once; a call may then fail with its error or give the right
values, never wrong ones."""
import numpy as np
import pytest

from test_gpu_parity import ctx  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu

WTB_ERR_EIG = 8


@pytest.fixture
def hasty():
    """a context whose waits give up after one poll"""
    from wantibexos_amd import bse
    with bse.Context(0) as c:
        c.set_wait_limit(1)
        yield c


def case(n1, n2):
    from wantibexos_amd import bse, tbmodel
    m = tbmodel.hex2d(seed=9, nw=6, ngrid=(12, 12, 1))
    return m, bse.BSEParams(ngrid=(n1, n2, 1), nc=2, nv=2, coultype="V2DRK", r0=40.0, cshift=0.05, ebse0=0.0,
                            ebsef=6.0, numbse=101, dtfull=True, cpol=True, f154=False)


# N = 4: the chase's only group of sweeps waits in LDS alone; 32: no panel at band 32; 144:
# one workgroup a panel; 576: three
@pytest.mark.parametrize("band", [16, 32])
@pytest.mark.parametrize("grid", [(1, 1), (2, 4), (6, 6), (12, 12)])
def test_stalled_plan_gives_no_wrong_values(ctx, hasty, grid, band):  # noqa: F811
    from wantibexos_amd import bse
    print(f"stalled plan {grid} band {band}", flush=True)
    m, prm = case(*grid)
    with bse.BSEPlan(ctx, m, prm) as plan:
        plan.set_reduction(False)
        plan.execute()
        ref = plan.results()
    with bse.BSEPlan(hasty, m, prm) as plan:
        plan.set_reduction(True, band)
        plan.execute()
        try:
            got = plan.results()
        except bse.WTBError as e:
            assert e.code == WTB_ERR_EIG
            return
    assert np.abs(got["W"] - ref["W"]).max() < 1e-12
    assert np.abs(got["eps"] - ref["eps"]).max() <= 1e-9 * np.abs(ref["eps"]).max()


def test_lowest_after_a_stalled_call(ctx):  # noqa: F811
    """the solver's buffers live on in the plan; a stall of one call is not the next one's"""
    from wantibexos_amd import bse
    m, prm = case(12, 12)
    prm.precision = bse.MIXED
    with bse.BSEPlan(ctx, m, prm) as plan:
        ref = plan.lowest(nev=16, tol=1e-8)["W"]
    with bse.Context(0) as c, bse.BSEPlan(c, m, prm) as plan:
        c.set_wait_limit(1)
        try:
            assert np.abs(plan.lowest(nev=16, tol=1e-8)["W"] - ref).max() < 1e-12
        except bse.WTBError as e:
            assert e.code == WTB_ERR_EIG
        c.set_wait_limit(0)
        assert np.abs(plan.lowest(nev=16, tol=1e-8)["W"] - ref).max() < 1e-12


# N = 36, 576: with any wait given up the one-stage form gives the values, to the bit
@pytest.mark.parametrize("grid", [(3, 3), (12, 12)])
def test_stalled_plan_is_solved_by_the_one_stage_form(ctx, hasty, grid):  # noqa: F811
    from wantibexos_amd import bse
    m, prm = case(*grid)
    with bse.BSEPlan(ctx, m, prm) as plan:
        plan.set_reduction(False)
        plan.execute()
        ref = plan.results()
    with bse.BSEPlan(hasty, m, prm) as plan:
        for _ in range(2):
            plan.execute()
            got = plan.results()
            for k in ("W", "act", "eps"):
                assert np.array_equal(got[k], ref[k]), k
    with bse.BSEBatch(hasty, [m, m], [prm, prm], lanes=2) as batch:
        batch.execute()
        for i in range(2):
            got = batch.results(i)
            for k in ("W", "act", "eps"):
                assert np.array_equal(got[k], ref[k]), k


@pytest.mark.parametrize("n", [40, 300])
def test_stalled_zheev_is_solved(hasty, n):
    from wantibexos_amd import bse
    rng = np.random.default_rng(n)
    a = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    a = a + a.conj().T
    w = bse.zheev(hasty, np.triu(a))
    assert np.linalg.norm(w - np.linalg.eigvalsh(a)) <= 8 * n * np.finfo(float).eps * np.linalg.norm(a)


@pytest.mark.parametrize("lanes", [1, 3])
def test_stalled_bands_are_solved(ctx, hasty, lanes):  # noqa: F811
    from wantibexos_amd import bse
    m, prm = case(6, 6)
    q = np.array([[0.0, 0.0, 0.0, 0.0], [0.1, 0.05, 0.0, 0.0], [0.2, 0.1, 0.02, 0.0], [0.3, 0.1, 0.1, 0.0]])
    with bse.BSEBands(ctx, m, prm, lanes=lanes) as b:
        ref = b.run(q)
    with bse.BSEBands(hasty, m, prm, lanes=lanes) as b:
        got = b.run(q)
    assert np.abs(got - ref).max() < 1e-12


def test_stalled_lowest_is_solved(ctx, hasty):  # noqa: F811
    from wantibexos_amd import bse
    m, prm = case(12, 12)
    prm.precision = bse.MIXED
    with bse.BSEPlan(ctx, m, prm) as plan:
        ref = plan.lowest(nev=16, tol=1e-8)["W"]
    with bse.BSEPlan(hasty, m, prm) as plan:
        assert np.abs(plan.lowest(nev=16, tol=1e-8)["W"] - ref).max() < 1e-12


def test_the_launches_of_eight_streams(ctx):  # noqa: F811
    """eight lanes at once, panels of one and of three workgroups"""
    from wantibexos_amd import bse
    for grid in ((6, 6), (12, 12)):
        m, prm = case(*grid)
        q = np.stack([np.linspace(0.0, 0.5, 16)] * 2 + [np.linspace(0.0, 0.2, 16), np.zeros(16)], axis=1)
        with bse.BSEBands(ctx, m, prm, lanes=1) as b:
            ref = b.run(q)
        with bse.BSEBands(ctx, m, prm, lanes=8) as b:
            for _ in range(3):
                assert np.array_equal(b.run(q), ref), grid


@pytest.mark.parametrize("bits", [0xFFFFFFFFFFFFFFFF, 0x7FF8000000000000])
def test_nan_of_any_bits_does_not_stall(ctx, bits):  # noqa: F811
    """an empty slot of the panels' exchange is a NaN of all ones; one in the matrix is a value
    like another (a wait that ran out would take most of a second and then the one-stage form)"""
    import time
    from wantibexos_amd import bse
    n = 300
    a = np.eye(n, dtype=complex)
    bse.zheev(ctx, a)
    a.view(np.uint64)[40, 2 * 100] = bits
    t = time.perf_counter()
    try:
        bse.zheev(ctx, a)
    except bse.WTBError as e:
        assert e.code == 10                     # NaN or Inf in the input
    assert time.perf_counter() - t < 0.2
