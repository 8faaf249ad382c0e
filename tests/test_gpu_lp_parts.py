"""BF16x3's operand in two and in four parts, and a plan that changes its precision."""
import numpy as np
import pytest

from test_gpu_gemm64 import krp, unfold

pytestmark = pytest.mark.gpu


def parts(x):
    """x = hi + lo in bfloat16 parts (round to nearest even) of its float32 value."""
    def bf(v):
        u = v.astype(np.float32).view(np.uint32)
        u = (u + 0x7FFF + ((u >> 16) & 1)) & np.uint32(0xFFFF0000)
        return u.view(np.float32)
    x = x.astype(np.float32)
    hi = bf(x)
    return hi.astype(np.float64), bf(x - hi).astype(np.float64)


# sides of two and three modes, ragged and one below, at and above a 32-index stage; ranks of
# one to three and of more blocks
CASES = [((5, 6, 7), 3), ((31, 7, 40), 16), ((32, 9, 30), 17), ((33, 30, 9, 8), 47), ((12, 11, 13, 10), 33),
         ((6, 5, 4, 3, 7), 20), ((40, 30, 20), 70)]


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("dims,R", CASES)
def test_products_of_the_rounded_factor(itcpd, dims, R, dt):
    """Each side's first M is that of the leading factor's two parts, T_hi (a_hi + a_lo) w +
    T_lo a_hi w, within the sums' rounding: 128 FP32 additions of up to five products, the
    weight's 2^-24 and 2^-24 of a product beyond its parts."""
    rng = np.random.default_rng(41)
    T = np.asfortranarray(rng.standard_normal(dims).astype(dt))
    fac = [rng.standard_normal((d, R)) for d in dims]
    sums = [np.prod(dims[:k]) + np.prod(dims[k:]) for k in range(1, len(dims))]
    s = max(k for k in range(1, len(dims)) if sums[k - 1] == min(sums))
    Th, Tl = parts(T)
    with itcpd.ALSPlan(T, R, prec="bf16x3") as plan:
        plan.set_cpd(itcpd.CPD(fac, np.ones(R)))
        for n, side in ((0, range(s, len(dims))), (s, range(s))):
            hi, lo = list(fac), list(fac)
            hi[side[0]], lo[side[0]] = parts(fac[side[0]])
            others = [m for m in range(len(dims)) if m != n]
            kh, kl = (krp([f[m] for m in others]) for f in (hi, lo))
            ref = unfold(Th, n) @ (kh + kl) + unfold(Tl, n) @ kh
            bound = (5 * 128 + 8) * 2.0**-24 * (np.abs(unfold(T.astype(np.float64), n)) @ np.abs(kh + kl))
            assert (np.abs(plan.mttkrp(n) - ref) / bound).max() <= 1.0, n


@pytest.mark.parametrize("order", [("fp32", "bf16x3"), ("bf16x3", "fp32"), ("fp64", "fp32", "bf16x3", "fp64")])
@pytest.mark.parametrize("dims,R", [((64, 64, 64, 64), 48), ((33, 30, 9, 8), 47), ((40, 30, 20), 70)])
def test_a_plan_that_changes_its_precision(itcpd, dims, R, order):
    """The same M as a plan of that precision from the start (a sum may be split otherwise): its
    buffers hold every form's operands."""
    rng = np.random.default_rng(42)
    T = np.asfortranarray(rng.standard_normal(dims).astype(np.float32))
    cp = itcpd.CPD([rng.standard_normal((d, R)) for d in dims], np.ones(R))
    with itcpd.ALSPlan(T, R, prec=order[0]) as plan:
        plan.set_cpd(cp)
        for prec in order:
            plan.set_precision(prec)
            with itcpd.ALSPlan(T, R, prec=prec) as fresh:
                fresh.set_cpd(cp)
                for n in range(len(dims)):
                    a, b = plan.mttkrp(n), fresh.mttkrp(n)
                    assert np.abs(a - b).max() <= 1e-5 * np.abs(b).max(), (prec, n)
