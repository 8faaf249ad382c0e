"""The reduced-precision GEMMs at the sizes where their tiles, stages and splits end and on
both sides of the rule between the LDS ring and the direct form."""
import numpy as np
import pytest

from test_gpu_gemm64 import krp, unfold

pytestmark = pytest.mark.gpu

SHAPES = [((64, 64, 64), 16), ((65, 63, 33), 17), ((63, 65, 31), 33), ((17, 15, 400), 48), ((400, 16, 3), 49),
          ((3, 5, 2), 1), ((50, 60), 7), ((300, 7), 65), ((33, 20, 17), 81), ((40, 30, 20), 150),
          ((16, 15, 14, 13), 32), ((2, 3, 5, 7, 11), 9), ((256, 256, 32), 80), ((64, 64, 64, 64), 48),
          ((64, 64, 64, 64), 32)]


@pytest.mark.parametrize("prec", ["fp32", "bf16x3"])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("dims,R", SHAPES)
def test_mttkrp_within_rounding_of_its_sums(itcpd, dims, R, dt, prec):
    """FP32: both operands rounded (2^-24 each; an FP32 tensor is exact), FP32 sums of at most
    128 products before they go to FP64.  BF16x3: |x - hi - lo| <= 2^-18 |x| per operand and
    the dropped lo lo <= 2^-18 of the product, on the same sums (of three products each)."""
    rng = np.random.default_rng(17)
    T = np.asfortranarray(rng.standard_normal(dims).astype(dt))
    cp = itcpd.CPD([rng.standard_normal((d, R)) for d in dims], np.ones(R))
    eps = (128 + 5) * 2.0**-24 if prec == "fp32" else 3 * 2.0**-18 + (3 * 128 + 5) * 2.0**-24
    with itcpd.ALSPlan(T, R, prec=prec) as plan:
        plan.set_cpd(cp)
        for n in range(len(dims)):
            K = krp([cp.factors[m] for m in range(len(dims)) if m != n])
            U = unfold(T.astype(np.float64), n)
            assert (np.abs(plan.mttkrp(n) - U @ K) / (eps * (np.abs(U) @ np.abs(K)))).max() <= 1.0, n


@pytest.mark.parametrize("prec", ["fp32", "bf16x3"])
@pytest.mark.parametrize("dims,at", [((37, 21, 18), (36, 20, 17)), ((37, 21, 18), (0, 0, 0)), ((20, 70, 5), (19, 69, 4))])
def test_non_finite_entries_stay_in_their_rows(itcpd, dims, at, prec):
    rng = np.random.default_rng(18)
    T = np.asfortranarray(rng.standard_normal(dims).astype(np.float32))
    T[at] = np.nan
    cp = itcpd.CPD([rng.standard_normal((d, 6)) for d in dims], np.ones(6))
    with itcpd.ALSPlan(T, 6, prec=prec) as plan:
        plan.set_cpd(cp)
        for n in range(3):
            bad = ~np.isfinite(plan.mttkrp(n)).all(axis=1)
            assert np.array_equal(np.nonzero(bad)[0], [at[n]])
