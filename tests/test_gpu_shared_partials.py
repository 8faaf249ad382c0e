"""Order-3 sweeps on partials shared across updates, with the form that ran told by its GEMM
launches: three for every two sweeps, the plain tree's two for each."""
import ctypes

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


# both splits of the plain tree; ranks whose factorisation rides along (R <= 64) and ranks above,
# where it is launched between the updates
@pytest.mark.parametrize("sweeps", [1, 2, 3, 4])
@pytest.mark.parametrize("dims,R", [((48, 40, 32), 5), ((33, 70, 90), 6), ((90, 91, 97), 17), ((160, 150, 170), 66),
                                    ((150, 151, 149), 80), ((190, 192, 180), 130)])
def test_shared_partials_run_and_match_the_oracle(itcpd, dims, R, sweeps):
    """Tolerance: the one of the plain tree's sweeps against the oracle."""
    rng = np.random.default_rng(61)
    true = [rng.standard_normal((d, R)) for d in dims]
    T = np.einsum("ir,jr,kr->ijk", *true, optimize=True) + 1e-3 * rng.standard_normal(dims)
    T = np.asfortranarray(T)
    init = O.random_CPD(T, R, np.random.default_rng(62))
    ref = O.als_optimize(T, init, check=O.NoCheck(sweeps), form="gemm")
    with itcpd.ALSPlan(T, R) as plan:
        plan.set_cpd(itcpd.CPD(init.factors, init.lam))
        plan.set_profiling(True)
        plan.run(itcpd.NoCheck(sweeps))
        gemms = plan.kernel_stats()["launches"]
        got = plan.get_cpd()
    assert gemms == (2 if sweeps == 1 else -(-3 * sweeps // 2))
    for a, b in zip(got.factors, ref.factors):
        assert np.linalg.norm(a - b) <= 1e-10 * np.linalg.norm(b)
    assert np.linalg.norm(got.lam - ref.lam) <= 1e-10 * np.linalg.norm(ref.lam)


def test_a_cube_needs_no_further_partial(itcpd):
    """The shared partial of equal modes is no larger than the plain tree's, which the run does
    not use: a run allocates nothing on the device."""
    hip = ctypes.CDLL("libamdhip64.so")

    def free():
        n, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(n), ctypes.byref(total)) == 0
        return n.value

    R = 48
    T = np.asfortranarray(np.random.default_rng(63).standard_normal((256, 256, 256)))
    init = itcpd.random_CPD(T, R, 64)
    used = []
    for _ in range(2):   # the first run loads the kernels
        with itcpd.ALSPlan(T, R) as plan:
            plan.set_cpd(init)
            plan.set_profiling(True)
            before = free()
            plan.run(itcpd.NoCheck(4))
            used.append(before - free())
            assert plan.kernel_stats()["launches"] == 6
    assert used[1] == 0
