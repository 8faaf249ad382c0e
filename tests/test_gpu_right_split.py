"""The split of the FP64 right GEMM's ring form where its tiles meet the resident workgroups."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


WORKGROUPS = 4 * 256   # of the ring form resident at once: four per compute unit


@pytest.mark.parametrize("R", [33, 48])
@pytest.mark.parametrize("per", [1.0, 0.5, 1.5, 2.0])
def test_one_right_mode_of_whole_tiles(itcpd, per, R):
    """A matrix whose second mode has `per` tiles of 64 columns for every resident workgroup (the
    factorisation that may ride along takes one's place), one sweep against the oracle: a solve's
    8 R eps cond(V) on either side, V the Gram of the first mode's new factor."""
    dims = (64, 64 * int(per * WORKGROUPS))
    rng = np.random.default_rng(51)
    T = np.asfortranarray(rng.standard_normal((64, R)) @ rng.standard_normal((R, dims[1]))
                          + 1e-3 * rng.standard_normal(dims))
    init = O.random_CPD(T, R, np.random.default_rng(52))
    ref = O.als_optimize(T, init, check=O.NoCheck(1), form="gemm")
    got = itcpd.als_optimize(T, itcpd.CPD(init.factors, init.lam), check=itcpd.NoCheck(1))
    tol = 2 * 8 * R * 2.0**-53 * np.linalg.cond(ref.factors[0].T @ ref.factors[0])
    for a, b in zip(got.factors, ref.factors):
        assert np.linalg.norm(a - b) <= tol * np.linalg.norm(b)
    assert np.linalg.norm(got.lam - ref.lam) <= tol * np.linalg.norm(ref.lam)
