"""CPD transfer and run state of a plan: host factors move through a pinned mirror up to 8 MiB
and per factor above, and a run longer than the plan's own trace gets a trace of its own."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,rank", [((5, 4, 3), 1), ((7, 6, 5), 17), ((70000, 3, 2), 16), ((30, 20), 65)])
def test_cpd_round_trip(itcpd, dims, rank):
    rng = np.random.default_rng(3)
    with itcpd.ALSPlan(np.asfortranarray(rng.standard_normal(dims)), rank) as plan:
        for _ in range(2):
            cp = itcpd.CPD([np.asfortranarray(rng.standard_normal((d, rank))) for d in dims],
                           rng.standard_normal(rank))
            plan.set_cpd(cp)
            out = plan.get_cpd()
            assert all(np.array_equal(a, b) for a, b in zip(cp.factors, out.factors))
            assert np.array_equal(cp.lam, out.lam)


def test_trace_longer_than_the_plans(itcpd):
    rng = np.random.default_rng(4)
    T = np.asfortranarray(rng.standard_normal((2, 3, 2, 3)))
    init = itcpd.random_CPD(T, 2, np.random.default_rng(5))
    traces = {}
    with itcpd.ALSPlan(T, 2) as plan:
        for iters in (1030, 1024, 1500, 3):
            plan.set_cpd(init)
            check = itcpd.FitCheck(-1.0, iters, float(np.linalg.norm(T)))   # never converges
            traces[iters] = np.asarray(plan.run(check)["fits"])
    for iters, tr in traces.items():
        assert len(tr) == iters and np.all(np.isfinite(tr))
        assert np.array_equal(tr, traces[1500][:iters])
