"""Row solves with a V whose factors have nearly equal columns, as swamps of ALS have them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = 2.0**-53


def triples(R, place):
    """Two groups of three columns: at the front, spread with the last one late, across the halves,
    or two of 16 neighbours and one far off."""
    return {"front": ((0, 1, 2), (3, 4, 5)), "spread": ((0, R // 3, R - 1), (1, R // 2, R - 2)),
            "inner": ((2, R // 3, R // 2), (R // 4, R // 2 + 1, R - 3)),
            "pairs": ((0, min(8, R - 4), min(40, R - 3)), (1, min(9, R - 2), R - 1))}[place]


def near_factors(R, near, unit, place, seed):
    rng = np.random.default_rng(seed)
    fac = [rng.standard_normal((R + 40, R)) for _ in range(2)]
    for f in fac:
        for a, b, c in triples(R, place):
            f[:, b] = f[:, a] + near * rng.standard_normal(R + 40)
            f[:, c] = f[:, a] + near * rng.standard_normal(R + 40)
        if unit:
            f /= np.linalg.norm(f, axis=0)
    return fac, rng


# unit columns as the sweeps have them, near 3e-3: lambda_min a few times the pivot tolerance,
# cond(V) 1e6 .. 4e6; columns as given: 1e5 .. 3e9
@pytest.mark.parametrize("place", ["front", "spread", "inner", "pairs"])
@pytest.mark.parametrize("unit,near", [(True, 1e-1), (True, 3e-3), (False, 1e-2), (False, 1e-4)])
@pytest.mark.parametrize("R", [10, 11, 16, 17, 32, 33, 37, 63, 64, 65, 100, 128, 129, 150, 193])
def test_solves_of_near_equal_columns(itcpd, R, unit, near, place):
    """X from M = X V.  A backward stable solve is within c R eps cond(V) ||X||, c = 8 as for
    well-conditioned V; M's rounding and V's (a Gram product on either side) are of that size."""
    fac, rng = near_factors(R, near, unit, place, 17)
    T = np.asfortranarray(rng.standard_normal((R + 40, R + 40, 12)))
    V = (fac[0].T @ fac[0]) * (fac[1].T @ fac[1])
    X = rng.standard_normal((12, R))
    with itcpd.ALSPlan(T, R) as plan:
        plan.set_cpd(itcpd.CPD(fac + [rng.standard_normal((12, R))], np.ones(R)))
        got, fell = plan.solve_ls(2, X @ V)
    assert not fell
    assert np.linalg.norm(got - X) <= 8 * R * EPS * np.linalg.cond(V) * np.linalg.norm(X)
