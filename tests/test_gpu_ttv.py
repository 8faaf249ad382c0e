"""The Hadamard-reduce of a dimension-tree side to its modes, at the lengths where its lanes,
batches of loads and splits end."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# sides whose other modes flatten to one below, at and above 64, 128, 192, 256 and 320
# elements (steps and batches of the wave), modes of one element, row groups with a rest, and
# leading modes with 1, 7, 8, 9 and several splits' worth of others
CASES = [((63, 5, 64, 5), 3), ((65, 4, 127, 3), 2), ((128, 7, 129, 6), 5), ((192, 2, 193, 1), 4),
         ((255, 9, 256, 10), 1), ((257, 3, 321, 2), 17), ((200, 13, 5, 13), 24), ((300, 8, 4, 16), 33),
         ((300, 1, 9, 7), 6), ((7, 1, 1, 2, 5), 3), ((23, 21, 20, 19, 18), 24), ((3, 2, 3, 2, 3, 2, 3), 8),
         ((5, 8, 6, 9), 70), ((400, 3, 40, 17, 2), 11)]


@pytest.mark.parametrize("dims,R", CASES)
def test_every_mode_within_rounding_of_its_sums(itcpd, dims, R):
    """|M - exact| <= (K + 2 N + 2) 2^-53 sum |T| |KRP| entry by entry, K the length of the
    sum: K - 1 additions in any order, and at most 2 N products of weights and terms."""
    rng = np.random.default_rng(11)
    T = np.asfortranarray(rng.standard_normal(dims))
    cp = itcpd.CPD([rng.standard_normal((d, R)) for d in dims], np.ones(R))
    with itcpd.ALSPlan(T, R) as plan:
        plan.set_cpd(cp)
        for n in range(len(dims)):
            krp = np.ones((1, R))
            for m in range(len(dims)):
                if m != n:
                    krp = (krp[:, None, :] * cp.factors[m][None]).reshape(-1, R)
            U = np.moveaxis(T, n, 0).reshape(dims[n], -1)
            bound = 2 * (U.shape[1] + 2 * len(dims) + 2) * 2.0**-53 * (np.abs(U) @ np.abs(krp))
            assert (np.abs(plan.mttkrp(n) - U @ krp) / bound).max() <= 1.0, n
