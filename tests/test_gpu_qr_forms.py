"""The column-pivoted QR of a sampled step in both of its forms, on samples that the corrected
normal equations do not certify."""
import numpy as np
import pytest

import oracle.sampled as S

pytestmark = pytest.mark.gpu

EPS = 2.0**-53


def uncertified(dims, R, ns):
    """Nearly equal columns: ||K^T K||_F ||(K^T K)^-1||_F >= cond(K)^2 far above the
    certificate's 1e8, so the QR solves."""
    rng = np.random.default_rng(71)
    fac = [rng.standard_normal((d, R)) for d in dims]
    for f in fac[1:]:
        f[:, R // 2] = f[:, 1] + 1e-6 * rng.standard_normal(f.shape[0])
    T = np.asfortranarray(rng.standard_normal(dims))
    smp = np.asfortranarray(np.stack([rng.integers(0, d, ns) for d in dims[1:]], axis=1).astype(np.int32))
    K = S.pivot_hadamard(fac[1:], smp)
    assert np.linalg.cond(K) >= 1e5
    return T, fac, smp, K


# the apply step in registers (ns <= 2048) and from memory; ranks on both sides of 64
@pytest.mark.parametrize("dims,R,ns", [((40, 30, 20), 12, 700), ((40, 30, 20), 12, 1500), ((25, 70, 60), 12, 2500),
                                       ((30, 60, 50), 48, 2048), ((30, 60, 50), 48, 2049), ((30, 60, 50), 70, 1500)])
def test_qr_forms_give_the_same_bits_and_least_squares(itcpd, dims, R, ns):
    """The one-workgroup form and the grid-wide steps agree bit for bit, and with least squares
    within 2 c eps (cond + cond^2 rho), c = 8 ns, rho the residual over ||K|| ||X||."""
    T, fac, smp, K = uncertified(dims, R, ns)
    out = []
    for rows in (0, 1 << 30):
        with itcpd.ALSPlan(T, R) as plan:
            plan.set_cpd(itcpd.CPD(fac, np.ones(R)))
            plan.set_qr_forms(4096, rows)
            assert plan.sampled_solve(0, smp, False)[1] == R
            got = plan.get_cpd()
            out.append(got.factors[0] * got.lam)
    assert np.array_equal(out[0], out[1])
    B = S.fused_flatten_sample(T, 0, smp).T
    ref = np.linalg.lstsq(K, B, rcond=None)[0]
    c, nK = np.linalg.cond(K), np.linalg.norm(K, 2)
    rho = np.linalg.norm(B - K @ ref) / (nK * np.linalg.norm(ref))
    assert np.linalg.norm(out[0].T - ref) <= 2 * 8 * ns * EPS * (c + c * c * rho) * np.linalg.norm(ref)
