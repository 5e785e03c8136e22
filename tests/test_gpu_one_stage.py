"""GPU: what the one-stage reduction still serves: panel widths and their tuner, and the lockstep
groups of a batch in both element types (FP64 plans of 32 rows on take the two-stage form unless
told otherwise)."""
import numpy as np
import pytest

from test_gpu_parity import ctx  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


def params(n1, n2, **kw):
    from wantibexos_amd import bse
    return bse.BSEParams(ngrid=(n1, n2, 1), nc=2, nv=2, coultype="V2DRK", r0=40.0, cshift=0.05, ebse0=0.0,
                         ebsef=6.0, numbse=101, dtfull=True, cpol=True, f154=False, **kw)


def model():
    from wantibexos_amd import tbmodel
    return tbmodel.hex2d(seed=9, nw=6, ngrid=(12, 12, 1))


def test_panel_widths(ctx):  # noqa: F811
    from wantibexos_amd import bse
    res = {}
    with bse.BSEPlan(ctx, model(), params(12, 12)) as plan:
        plan.set_reduction(False)
        for nb in (16, 20, 24, 32):
            plan.set_panel(nb)
            plan.execute()
            res[nb] = plan.results()
        best, ms = plan.tune()
        plan.execute()
        tuned = plan.results()
    assert best in (16, 20, 24, 32) and all(t > 0 for t in ms.values())
    for nb in (16, 20, 24):
        assert np.abs(res[nb]["W"] - res[32]["W"]).max() < 1e-11
        assert not np.array_equal(res[nb]["act"], res[32]["act"])     # another grouping of the updates
    assert np.array_equal(tuned["W"], res[best]["W"]) and np.array_equal(tuned["act"], res[best]["act"])


def test_nothing_to_tune(ctx):  # noqa: F811
    """the two-stage form has no panels of a chosen width"""
    from wantibexos_amd import bse
    with bse.BSEPlan(ctx, model(), params(12, 12)) as plan:
        plan.set_panel(20)
        best, ms = plan.tune()
        assert best == 20 and all(t == 0 for t in ms.values())
    with bse.BSEBatch(ctx, [model()] * 2, [params(6, 6), params(6, 6, precision=bse.MIXED)]) as b:
        t = b.tune()
        assert t[0] == 32 and t[1] in (16, 20, 24, 32)


@pytest.mark.parametrize("lanes", [1, 3])
def test_lockstep_groups(ctx, lanes):  # noqa: F811
    """FP64 below 32 rows, the precision form at several sizes: as the plans alone, to the bit"""
    from wantibexos_amd import bse
    m = model()
    prms = [params(*g) for g in [(1, 1), (1, 5), (1, 7), (2, 3)]]
    prms += [params(*g, precision=bse.MIXED) for g in [(1, 5), (3, 4), (6, 6), (12, 12)]]
    with bse.BSEBatch(ctx, [m] * len(prms), prms, lanes=lanes) as b:
        for _ in range(2):
            b.execute()
            for i, p in enumerate(prms):
                with bse.BSEPlan(ctx, m, p) as plan:
                    plan.execute()
                    ref = plan.results()
                got = b.results(i)
                for k in ("W", "act", "eps"):
                    assert np.array_equal(got[k], ref[k]), (i, k)


def test_kernel_times_are_those_of_the_form_that_ran(ctx):  # noqa: F811
    from wantibexos_amd import bse
    with bse.BSEPlan(ctx, model(), params(12, 12)) as plan:
        plan.set_timing(2)
        seen = []
        for form in (False, None, False, None):
            plan.set_reduction(form)
            plan.execute()
            plan.results()
            seen.append((plan.kernel_ms()[1], plan.kernel_flops() > 0))
    # 575 GEMVs; 35 panels of 16 columns
    assert seen == [(575, False), (35, True)] * 2
