"""The memory form of the ACA (ranks above 64, Matern kernels): one wavefront, four and eight
per block give the oracle's ranks and product."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


# a tolerance, or a rank bound well below the blocks' numerical ranks, so that no rank is
# decided at rounding level: the oracle's ranks stay as they are and its products move by less
# than 5e-12 when its length scale changes by one or two bits.  1e-8: the FP64 products' bar
@pytest.mark.parametrize("kind,dim,k,n,tol", [(O.K_EXPONENTIAL, 2, 80, 3000, 1e-6), (O.K_MATERN_REF, 2, 16, 6000, 0.0),
                                              (O.K_EXPONENTIAL, 3, 70, 3000, 1e-6)])
def test_teams_of_the_memory_form(gpu, kind, dim, k, n, tol):
    X = O.uniform(8600 + n, dim * n).reshape(dim, n)
    hm = gpu.HMatrix(X, X, 32 if dim == 2 else 20, 1.0, 50, 96, k, epsilon=max(tol, 1e-6))
    hm.set_option(gpu.OPT_ACA_TOLERANCE, 2 if tol else 0)
    hm.setup()
    kern = gpu.Kernel(kind, 0.0, 1.0)
    hm.set_kernel(kern)
    om = O.HMatrix(X, X, 32 if dim == 2 else 20, 1.0, 50, 96)
    ok = O.kernel(kind, dim, 0.0, 1.0)
    om.aca(ok, k, tol_mode=2 if tol else 0, eps=tol)
    f = om.aca_factors()
    b = hm.blocks(O.WORK_ITEM_DTYPE)
    b = b[b["work_type"] == gpu.WT_ACA]
    size = (b["set1_u"] - b["set1_l"]) + (b["set2_u"] - b["set2_l"]) + 2
    mem = size[f["kb"] > 64] if k > 64 else size
    assert len(mem) > 10
    x = O.normal(8700 + n, n)
    ref = om.hmvp(ok, x)
    lo, hi = int(np.quantile(mem, 0.3)), int(np.quantile(mem, 0.7))
    y = []
    # (workgroups of 4 above .., of 8 above ..): by size, all on one wavefront, on 4, on 8
    for big, huge in ((lo, hi), (1 << 30, 1 << 30), (0, 1 << 30), (0, 0)):
        hm.set_option(gpu.OPT_ACA_BIG_BLOCK, big)
        hm.set_option(gpu.OPT_ACA_HUGE_BLOCK, huge)
        for scan in (0, 1):
            hm.set_option(gpu.OPT_ACA_ROW_SCAN, scan)
            hm.precompute_aca()
            assert hm.work()["rank_sum"] == int(f["keff"].sum())
            y.append(hm.apply(x))
            assert np.linalg.norm(y[-1] - ref) <= 1e-8 * np.linalg.norm(ref)
        np.testing.assert_array_equal(y[-1], y[-2])
    hm.destroy()
    kern.free()
