"""GPU: the COMPLEX*16 two-stage reductions of a batch in shared launches: every matrix to the
bit as in its own plan, whatever runs beside it."""
import numpy as np
import pytest

from test_gpu_parity import ctx  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


def params(n1, n2, **kw):
    from wantibexos_amd import bse
    return bse.BSEParams(ngrid=(n1, n2, 1), nc=2, nv=2, coultype="V2DRK", r0=40.0, cshift=0.05, ebse0=0.0,
                         ebsef=6.0, numbse=101, dtfull=True, cpol=True, f154=False, **kw)


def single(ctx, m, p):
    from wantibexos_amd import bse
    with bse.BSEPlan(ctx, m, p) as plan:
        plan.execute()
        return plan.results()


def check(ctx, m, prms, lanes, repeat=2):
    from wantibexos_amd import bse
    ref = {}
    with bse.BSEBatch(ctx, [m] * len(prms), prms, lanes=lanes) as b:
        for _ in range(repeat):               # the first execute captures, the others replay
            b.execute()
            for i, p in enumerate(prms):
                key = (p.ngrid, p.precision, p.bset)
                if key not in ref:
                    ref[key] = single(ctx, m, p)
                got = b.results(i)
                for k in ("W", "act", "eps"):
                    assert np.array_equal(got[k], ref[key][k]), (lanes, i, p.ngrid, k)


# N = 20: one-stage, FP64 lockstep; 32: one panel; 48, 52: panels end; 272 | 276: one and two
# workgroups a panel; 1024: several; 2704: on a lane of its own; the precision form's
# lockstep and finite temperature's six tracked vectors beside them
@pytest.mark.parametrize("lanes", [1, 3])
def test_uneven_set(ctx, lanes):  # noqa: F811
    from wantibexos_amd import bse, tbmodel
    m = tbmodel.hex2d(seed=9, nw=6, ngrid=(12, 12, 1))
    print(f"uneven set, lanes {lanes}", flush=True)
    prms = [params(*g) for g in [(1, 5), (2, 4), (3, 4), (1, 13), (4, 17), (3, 23), (16, 16), (1, 5), (26, 26)]]
    prms += [params(6, 6, precision=bse.MIXED), params(3, 4, precision=bse.MIXED)]
    prms += [params(6, 6, bset=True, temp=3000.0, ta="VE", st=0.3, phavg=0.05)]
    check(ctx, m, prms, lanes)


# more members than a launch takes, and more panel workgroups (70 x 5)
@pytest.mark.parametrize("grid", [(3, 3), (13, 20)])
def test_more_members_than_a_launch(ctx, grid):  # noqa: F811
    from wantibexos_amd import tbmodel
    m = tbmodel.hex2d(seed=9, nw=6, ngrid=(12, 12, 1))
    print(f"70 members of {grid}", flush=True)
    check(ctx, m, [params(*grid)] * 70, 4)


def test_stalled_set_is_solved_by_the_one_stage_form(ctx):  # noqa: F811
    from wantibexos_amd import bse, tbmodel
    m = tbmodel.hex2d(seed=9, nw=6, ngrid=(12, 12, 1))
    prms = [params(*g) for g in [(3, 3), (6, 6), (12, 12), (2, 4)]]
    with bse.Context(0) as hasty:
        hasty.set_wait_limit(1)
        with bse.BSEBatch(hasty, [m] * 4, prms, lanes=2) as b:
            for _ in range(2):
                b.execute()
                for i, p in enumerate(prms):
                    with bse.BSEPlan(ctx, m, p) as plan:
                        plan.set_reduction(False)
                        plan.execute()
                        ref = plan.results()
                    got = b.results(i)
                    for k in ("W", "act", "eps"):
                        assert np.array_equal(got[k], ref[k]), (i, k)
