"""The sampled step's least squares by corrected normal equations, at the edges of its tiles and
16-sample chunks, and the column-pivoted QR behind its certificate; leverage scores by blocks."""
import numpy as np
import pytest

import oracle.sampled as S

pytestmark = pytest.mark.gpu

EPS = 2.0**-53


def step(itcpd, T, fac, mode, smp, form=None):
    R = fac[0].shape[1]
    with itcpd.ALSPlan(T, R) as plan:
        plan.set_cpd(itcpd.CPD(fac, np.ones(R)))
        if form is not None:
            plan.set_qr_forms(4096, form)
        plan.sampled_solve(mode, smp, False)
        got = plan.get_cpd()
    return got.factors[mode] * got.lam


def problem(dims, R, ns, mode, dt=np.float64, near=None):
    rng = np.random.default_rng(31)
    T = np.asfortranarray(rng.standard_normal(dims).astype(dt))
    fac = [rng.standard_normal((d, R)) for d in dims]
    if near is not None:
        for f in fac:
            f[:, 1] = f[:, 0] + near * f[:, 1]
    smp = np.asfortranarray(np.stack([rng.integers(0, d, ns) for m, d in enumerate(dims) if m != mode], axis=1)
                            .astype(np.int32))
    K = S.pivot_hadamard([f for m, f in enumerate(fac) if m != mode], smp)
    B = S.fused_flatten_sample(T.astype(np.float64), mode, smp)
    return T, fac, smp, K, B


def bound(K, B, X):
    """Least squares, backward stable: relative forward error within c eps (cond + cond^2 rho),
    rho = ||residual|| / (||K|| ||X||), here with c = 8 ns for either side."""
    c, nK = np.linalg.cond(K), np.linalg.norm(K, 2)
    rho = np.linalg.norm(B - K @ X) / (nK * np.linalg.norm(X))
    return 2 * 8 * K.shape[0] * EPS * (c + c * c * rho)


def least_squares(K, B):
    return B.T, np.linalg.lstsq(K, B.T, rcond=None)[0]


CASES = [((5, 6, 7), 1, 1, 0), ((15, 9, 8), 5, 15, 0), ((16, 9, 8), 5, 16, 0), ((17, 12, 11), 16, 40, 0),
         ((9, 33, 20), 17, 127, 1), ((30, 20, 31), 31, 128, 2), ((40, 30, 20), 32, 129, 0), ((30, 40, 50), 33, 300, 2),
         ((20, 64, 50), 49, 257, 1), ((65, 40, 50), 64, 1000, 0), ((14, 13, 12, 11), 20, 513, 2)]


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("dims,R,ns,mode", CASES)
def test_step_within_least_squares_bound(itcpd, dims, R, ns, mode, dt):
    T, fac, smp, K, B = problem(dims, R, ns, mode, dt)
    X = step(itcpd, T, fac, mode, smp)
    B, ref = least_squares(K, B)
    assert np.linalg.norm(X.T - ref) <= bound(K, B, ref) * np.linalg.norm(ref)


@pytest.mark.parametrize("near", [3e-2, 1e-3, 1e-5])
@pytest.mark.parametrize("dims,R,ns,mode", [((40, 30, 20), 12, 400, 0), ((20, 64, 50), 40, 700, 1)])
def test_ill_conditioned_samples(itcpd, dims, R, ns, mode, near):
    """Nearly equal columns, on both sides of the certificate (cond(K) from about 50 to past
    1e5, where the QR solves): the same bound, and both forms of the QR agree bit for bit."""
    T, fac, smp, K, B = problem(dims, R, ns, mode, near=near)
    X = step(itcpd, T, fac, mode, smp, 0)
    B, ref = least_squares(K, B)
    assert np.linalg.norm(X.T - ref) <= bound(K, B, ref) * np.linalg.norm(ref)
    assert np.array_equal(X, step(itcpd, T, fac, mode, smp, 1 << 30))


@pytest.mark.parametrize("rows", [64, 65, 79, 80, 130])
@pytest.mark.parametrize("R", [1, 15, 16, 17, 32, 33, 48, 49, 63])
def test_leverage_scores_by_blocks(itcpd, rows, R):
    """p_i = ||q_i||^2 / R of a well-conditioned factor (cond below 100): error within
    8 R eps cond^2 of each score's bound 1."""
    rng = np.random.default_rng(32)
    Q, _ = np.linalg.qr(rng.standard_normal((rows, R)))
    A = Q * np.exp(rng.uniform(-1, 1, R))
    assert np.linalg.cond(A) < 10
    with itcpd.ALSPlan(np.asfortranarray(rng.standard_normal((rows, 3))), R) as plan:
        plan.set_cpd(itcpd.CPD([A, rng.standard_normal((3, R))], np.ones(R)))
        got = plan.leverage_scores(0)
    assert np.abs(got - (Q * Q).sum(axis=1) / R).max() <= 8 * R * EPS * 100
