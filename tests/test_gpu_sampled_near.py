"""Sampled least-squares steps on a low-rank tensor whose factors have nearly equal columns: no
residual hides the solve's error, on both sides of the corrected form's certificate."""
import numpy as np
import pytest

import oracle.sampled as S

pytestmark = pytest.mark.gpu

EPS = 2.0**-53


def problem(dims, R, ns, near):
    rng = np.random.default_rng(41)
    fac = [rng.standard_normal((d, R)) for d in dims]
    for f in fac[1:]:
        for a, b, c in ((0, 1, 2), (3, R // 2, R - 1)):
            f[:, b] = f[:, a] + near * rng.standard_normal(f.shape[0])
            f[:, c] = f[:, a] + near * rng.standard_normal(f.shape[0])
    T = np.asfortranarray(np.einsum("ir,jr,kr->ijk", *fac))
    smp = np.asfortranarray(np.stack([rng.integers(0, d, ns) for d in dims[1:]], axis=1).astype(np.int32))
    return T, fac, smp, S.pivot_hadamard(fac[1:], smp)


# cond(K) from 1e2 to 1e5; ||K^T K||_F ||(K^T K)^-1||_F passes the certificate's 1e8 on the way
@pytest.mark.parametrize("near", [1e-1, 1e-2, 1e-3, 5e-4, 3e-4, 1e-5])
@pytest.mark.parametrize("dims,R,ns", [((20, 40, 30), 10, 300), ((20, 40, 30), 16, 500), ((33, 30, 40), 24, 600),
                                       ((33, 30, 40), 32, 700), ((17, 60, 50), 47, 900), ((20, 70, 70), 64, 1100)])
def test_step_on_a_low_rank_tensor(itcpd, dims, R, ns, near):
    """The step's solution is the factor that the tensor was made of.  Backward stable least
    squares with no residual: within c eps cond(K), c = 8 ns for the solve and again for the
    rounding of T."""
    T, fac, smp, K = problem(dims, R, ns, near)
    with itcpd.ALSPlan(T, R) as plan:
        plan.set_cpd(itcpd.CPD([np.ones((dims[0], R))] + fac[1:], np.ones(R)))
        plan.sampled_solve(0, smp, False)
        got = plan.get_cpd()
    err = np.linalg.norm(got.factors[0] * got.lam - fac[0]) / np.linalg.norm(fac[0])
    assert err <= 2 * 8 * ns * EPS * np.linalg.cond(K)


@pytest.mark.parametrize("dims,R,ns", [((20, 40, 30), 10, 300), ((300, 40, 30), 10, 300), ((17, 60, 50), 47, 900),
                                       ((2100, 30, 40), 64, 1100)])
def test_uncertified_step_sets_the_whole_cpd(itcpd, dims, R, ns):
    """Equal columns: the corrected form leaves the CPD alone and the QR's solution sets factor,
    lambda and Gram, also on a new plan whose solution buffer holds nothing yet.  Rank and
    residual as least squares has them; V of mode 1 = G_0 .* G_2 within the rounding of its sums."""
    T, fac, smp, K = problem(dims, R, ns, 0.0)
    B = S.fused_flatten_sample(T, 0, smp)
    rank = np.linalg.matrix_rank(K)
    assert rank < R
    with itcpd.ALSPlan(T, R) as plan:
        plan.set_cpd(itcpd.CPD([np.ones((dims[0], R))] + fac[1:], np.ones(R)))
        info = plan.sampled_solve(0, smp, False)
        got = plan.get_cpd()
        V = plan.compute_krp(1)
    A, F = got.factors[0], fac[2]
    assert info[1] == rank
    assert np.linalg.norm(B.T - K @ (A * got.lam).T) <= 16 * ns * EPS * np.linalg.norm(K, 2) * np.linalg.norm(fac[0])
    bound = 2 * (dims[0] + dims[2] + 8) * EPS * (np.abs(A).T @ np.abs(A)) * (np.abs(F).T @ np.abs(F))
    assert (np.abs(V - (A.T @ A) * (F.T @ F)) / bound).max() <= 1.0
