"""The one-workgroup update of short modes, R <= 32: at one below, at and above its 16-row
tiles and the longest modes it takes (256 rows for R <= 16, 128 for R <= 32), next to the
separate launches."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

SHAPES = [((2, 3, 4), 1), ((15, 16, 17), 3), ((63, 64, 65), 15), ((255, 256, 257), 16), ((40, 127, 128), 17),
          ((129, 31, 33), 31), ((33, 49, 47), 32), ((60, 9, 8, 7), 6), ((9, 8, 7, 6, 5), 20), ((300, 18), 10)]


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def problem(dims, R, seed):
    rng = np.random.default_rng(seed)
    T = O.reconstruct([rng.standard_normal((d, R)) for d in dims], np.ones(R))
    T = np.asfortranarray(T + 1e-2 * np.linalg.norm(T) / np.sqrt(T.size) * rng.standard_normal(dims))
    return T, O.random_CPD(T, R, np.random.default_rng(seed + 1))


@pytest.mark.parametrize("kind", ["none", "fit", "diff"])
@pytest.mark.parametrize("dims,R", SHAPES)
def test_two_sweeps_match_oracle(itcpd, dims, R, kind):
    """Two sweeps of solves whose rounding grows by at most cond(V): 8 R 2^-53 cond(V) is
    below 1e-10 for these problems (cond(V) at most 630, at R = 10)."""
    T, init = problem(dims, R, 21)
    norm = float(np.linalg.norm(T))

    def checks(mod):
        return {"none": lambda: mod.NoCheck(2), "fit": lambda: mod.FitCheck(0.0, 2, norm),
                "diff": lambda: mod.CPDiffCheck(0.0, 2)}[kind]()

    ref = O.als_optimize(T, init, check=checks(O), form="gemm")
    check = checks(itcpd)
    got = itcpd.als_optimize(T, itcpd.CPD(init.factors, init.lam), check=check)
    for a, b in zip(got.factors, ref.factors):
        assert rel(a, b) <= 1e-10
    assert rel(got.lam, ref.lam) <= 1e-10


@pytest.mark.parametrize("dims,R", [((5, 6, 7), 2), ((17, 40, 33), 16), ((20, 120, 31), 32), ((250, 12, 18), 9)])
def test_deficient_rank_takes_the_qr_rows(itcpd, dims, R):
    """Two equal columns in every factor: each V is singular, the rows come from the QR path,
    and the equal columns stay equal."""
    T, init = problem(dims, R, 22)
    fac = [f.copy() for f in init.factors]
    for f in fac:
        f[:, 1] = f[:, 0]
    tr = {}
    ref = O.als_optimize(T, O.CPD(fac, init.lam), check=O.FitCheck(0.0, 1, float(np.linalg.norm(T))), form="gemm",
                         trace=tr)
    assert tr["fallbacks"] == 3
    got = itcpd.als_optimize(T, itcpd.CPD(fac, init.lam),
                             check=itcpd.FitCheck(0.0, 1, float(np.linalg.norm(T))))
    for a, b in zip(got.factors, ref.factors):
        assert rel(a, b) <= 1e-9
        assert rel(a[:, 1], a[:, 0]) <= 1e-9
