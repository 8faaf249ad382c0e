"""The direct FP64 GEMMs and the order-3 sweeps that share partials, at the sizes where
their tiles, stages and splits end."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def unfold(T, n):
    return np.moveaxis(T, n, 0).reshape(T.shape[n], -1)


def krp(fac):
    out = fac[0]
    for f in fac[1:]:
        out = (out[:, None, :] * f[None]).reshape(-1, f.shape[1])
    return out


# modes at and one off multiples of the 16-output tiles, 4- and 16-index steps; slabs smaller
# than a tile; one-element modes; orders whose Khatri-Rao product is formed whole, by rest
# weights and on the way; ranks around every block count
SHAPES = [((64, 64, 64), 16), ((65, 63, 33), 17), ((63, 65, 31), 33), ((17, 15, 400), 48), ((400, 16, 3), 49),
          ((3, 5, 2), 1), ((1, 40, 30), 4), ((40, 1, 30), 4), ((50, 60), 7), ((300, 7), 65), ((31, 29, 27), 80),
          ((33, 20, 17), 81), ((40, 30, 20), 150), ((16, 15, 14, 13), 32), ((2, 3, 5, 7, 11), 9),
          ((130, 3, 2, 2), 20), ((2, 2, 3, 130), 20), ((9, 8, 7, 6, 5), 64)]


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("dims,R", SHAPES)
def test_mttkrp_within_rounding_of_its_sums(itcpd, dims, R, dt):
    """Every entry within the rounding bound of a length-K FP64 dot product with N factors:
    (K + N + 2) 2^-53 sum |T| |KRP| for each side of the comparison (the FP32 tensor is exact
    in FP64)."""
    rng = np.random.default_rng(7)
    T = np.asfortranarray(rng.standard_normal(dims).astype(dt))
    cp = itcpd.CPD([rng.standard_normal((d, R)) for d in dims], np.ones(R))
    with itcpd.ALSPlan(T, R) as plan:
        plan.set_cpd(cp)
        for n in range(len(dims)):
            K = krp([cp.factors[m] for m in range(len(dims)) if m != n])
            U = unfold(T.astype(np.float64), n)
            bound = 2 * (U.shape[1] + len(dims) + 2) * 2.0**-53 * (np.abs(U) @ np.abs(K))
            assert (np.abs(plan.mttkrp(n) - U @ K) / bound).max() <= 1.0, n


@pytest.mark.parametrize("value", [np.inf, np.nan])
@pytest.mark.parametrize("dims,at", [((37, 21, 18), (36, 20, 17)), ((37, 21, 18), (0, 0, 0)), ((20, 70, 5), (19, 69, 4))])
def test_non_finite_entries_stay_in_their_rows(itcpd, dims, at, value):
    """Reads past the end take a valid element: one that is not finite reaches only the rows
    of M that it belongs to."""
    rng = np.random.default_rng(8)
    T = np.asfortranarray(rng.standard_normal(dims))
    T[at] = value
    cp = itcpd.CPD([rng.standard_normal((d, 6)) for d in dims], np.ones(6))
    with itcpd.ALSPlan(T, 6) as plan:
        plan.set_cpd(cp)
        for n in range(3):
            bad = ~np.isfinite(plan.mttkrp(n)).all(axis=1)
            assert np.array_equal(np.nonzero(bad)[0], [at[n]])


@pytest.mark.parametrize("sweeps", [1, 2, 3, 4])
@pytest.mark.parametrize("dims,R", [((48, 40, 32), 5), ((33, 70, 90), 6), ((90, 31, 47), 17), ((80, 81, 82), 66)])
def test_shared_partials_match_oracle(itcpd, dims, R, sweeps):
    """Odd and even numbers of sweeps (the last partial of an odd run serves one update), both
    splits of the plain tree, ranks with and without the factorisation riding along."""
    rng = np.random.default_rng(9)
    true = [rng.standard_normal((d, R)) for d in dims]
    T = np.einsum("ir,jr,kr->ijk", *true) + 1e-3 * rng.standard_normal(dims)
    init = O.random_CPD(T, R, np.random.default_rng(10))
    ref = O.als_optimize(T, init, check=O.NoCheck(sweeps), form="gemm")
    got = itcpd.als_optimize(T, itcpd.CPD(init.factors, init.lam), check=itcpd.NoCheck(sweeps))
    for a, b in zip(got.factors, ref.factors):
        assert np.linalg.norm(a - b) <= 1e-10 * np.linalg.norm(b)
    assert np.linalg.norm(got.lam - ref.lam) <= 1e-10 * np.linalg.norm(ref.lam)


@pytest.mark.parametrize("R", [1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 80, 127, 128, 129, 191, 192, 193, 257])
def test_inverse_solves(itcpd, R):
    """One wave (R <= 32), one workgroup (R <= 64) and two to five pivot blocks, the last of 1
    to 64 rows.  Forward error of an
    inverse-based solve: 8 R 2^-53 cond(V) of the solution's norm; and a V of deficient rank
    goes to the QR path."""
    rng = np.random.default_rng(11)
    dims = (R + 40, R + 30, 40)
    T = np.asfortranarray(rng.standard_normal(dims))
    fac = [rng.standard_normal((d, R)) / np.sqrt(d) for d in dims]
    with itcpd.ALSPlan(T, R) as plan:
        plan.set_cpd(itcpd.CPD(fac, np.ones(R)))
        M = rng.standard_normal((40, R))
        V = (fac[0].T @ fac[0]) * (fac[1].T @ fac[1])
        X, fell = plan.solve_ls(2, M)
        ref = np.linalg.solve(V, M.T).T
        assert not fell
        assert np.linalg.norm(X - ref) <= 8 * R * 2.0**-53 * np.linalg.cond(V) * np.linalg.norm(ref)
        if R == 1:
            return
        fac[0][:, 1], fac[1][:, 1] = fac[0][:, 0], fac[1][:, 0]
        plan.set_cpd(itcpd.CPD(fac, np.ones(R)))
        assert plan.solve_ls(2, M)[1]


@pytest.mark.parametrize("rows", [1, 15, 16, 17, 63, 2048, 2049, 5000])
@pytest.mark.parametrize("R", [1, 16, 17, 70])
def test_seeded_grams(itcpd, rows, R):
    """G_n = A_n^T A_n after set_cpd, through V of the modes of a two-mode tensor: the
    rounding bound of its sums."""
    rng = np.random.default_rng(12)
    A = [rng.standard_normal((rows, R)), rng.standard_normal((3, R))]
    with itcpd.ALSPlan(np.asfortranarray(rng.standard_normal((rows, 3))), R) as plan:
        plan.set_cpd(itcpd.CPD(A, np.ones(R)))
        for mode in (0, 1):
            B = A[1 - mode]
            bound = 2 * (B.shape[0] + 2) * 2.0**-53 * (np.abs(B).T @ np.abs(B))
            assert (np.abs(plan.compute_krp(mode) - B.T @ B) / bound).max() <= 1.0, mode
