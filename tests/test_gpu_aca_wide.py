"""Wide blocks of the ACA (more than 1024 rows or columns): their ranks and factors do not
depend on whether a long row search suspends the block, nor on the team that resumes it."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def _one_block(gpu, m1, m2, dim, k, ls=0.1):
    """Two point sets whose root block is the one admissible block.  In Morton order set 1
    begins with points too far from set 2 for any entry to count, a search of hundreds of rows."""
    X1 = 0.5 * O.uniform(8100 + m1, dim * m1).reshape(dim, m1)
    X2 = (0.9 if dim == 2 else 0.75) + 0.5 * O.uniform(8200 + m2, dim * m2).reshape(dim, m2)
    hm = gpu.HMatrix(X1, X2, 32 if dim == 2 else 20, 20.0, 50, 16, k)
    hm.setup()
    kern = gpu.Kernel(O.K_GAUSSIAN, 0.0, ls)
    hm.set_kernel(kern)
    assert hm.work()["aca"] == 1 and hm.work()["dense"] == 0
    return hm, kern


@pytest.mark.parametrize("m1,m2,dim", [(1500, 1300, 2), (3000, 2100, 2), (2000, 1100, 3), (9000, 2000, 2)])
def test_stop_of_a_suspended_block(gpu, m1, m2, dim):
    # the tolerance at which the stop comes one rank later, to the last bit, is the same
    # function of the factors with the row scan (the block is suspended and resumed) and without
    hm, kern = _one_block(gpu, m1, m2, dim, 24)
    hm.set_option(gpu.OPT_ACA_TOLERANCE, 2)

    def rank(scan, eps):
        hm.set_option(gpu.OPT_ACA_ROW_SCAN, scan)
        hm.data.epsilon = eps
        hm.precompute_aca()
        return hm.work()["rank_sum"]

    for target in (2, 5, 9):
        lo, hi = 1e-14, 1.0 - 1e-9  # rank(lo) > target >= rank(hi)
        assert rank(1, lo) > target >= rank(1, hi)
        while hi > np.nextafter(lo, 1.0):
            # halfway between their bit patterns
            a, b = np.float64(lo).view(np.int64), np.float64(hi).view(np.int64)
            mid = float(np.int64(a + (b - a) // 2).view(np.float64))
            lo, hi = (mid, hi) if rank(1, mid) > target else (lo, mid)
        assert rank(0, lo) > target >= rank(0, hi), (target, lo)
    hm.destroy()
    kern.free()
