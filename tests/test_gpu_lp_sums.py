"""How many products the direct FP32 GEMMs sum in FP32 before they go to FP64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("R", [3, 20, 40, 60])
def test_direct_sums_run_over_sixteen_indices(itcpd, R, mode, dt):
    """One 1 per 128 reduction indices among values of which four are below half a unit of its
    last place: an FP32 sum that has met the 1 loses the rest.  Sums of at most 16 products stay
    within (16 + 5) 2^-24 of the absolute sum; over 128 they are off by 30 2^-24."""
    dims = (650, 645)   # no multiple of the ring form's 256-row tiles
    idx = np.arange(dims[1 - mode])
    row = np.where(idx % 128 == 0, 1.0, 0.99 * 2.0**-26).astype(np.float32)
    T = np.empty(dims, dt, order="F")
    T[...] = row[None, :] if mode == 0 else row[:, None]
    with itcpd.ALSPlan(T, R, prec="fp32") as plan:
        plan.set_cpd(itcpd.CPD([np.ones((d, R)) for d in dims], np.ones(R)))
        got = plan.mttkrp(mode)
    want = row.astype(np.float64).sum()
    assert np.abs(got - want).max() <= (16 + 5) * 2.0**-24 * want
