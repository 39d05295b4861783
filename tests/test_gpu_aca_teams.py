"""The register form of the ACA at the edges of its team sizes: two point sets apart
from each other whose root block is the one admissible block, so that its numbers of
rows and columns are chosen freely."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

# The factors are formed as the oracle forms them, up to the last bits of exp and the
# order of the row norms.  Rows are taken in order, so a pivot may be small against the
# residual, and each such step magnifies the bits: the oracle's own product moves by up to
# 1e-5 here (2D, ranks of 24 and more) when its length scale changes by one or two bits,
# by less than 2e-11 in 3D.  Eight times what the oracle shows for four such changes, and
# no less than 1e-9.
TOL = 1e-9


def _bits(om, dim, k, tol, x, ref):
    d = []
    for e in (-2, -1, 1, 2):
        ok = O.kernel(O.K_EXPONENTIAL, dim, 0.0, 1.0 + e * 2.3e-16)
        om.aca(ok, k, tol_mode=2 if tol else 0, eps=tol)
        d.append(np.linalg.norm(om.hmvp(ok, x) - ref) / np.linalg.norm(ref))
    return max(d)


# edges of teams of 1, 2, 3, 4, 5, 8, 9, 12 and 16 wavefronts, of the wide blocks on 4
# and on 8, and ranks at the edges of the terms in registers (8, 16) and in LDS (16, 24)
@pytest.mark.parametrize("m1,m2,k", [
    (2, 70, 8), (64, 33, 7), (65, 64, 9), (128, 129, 16), (192, 5, 5), (193, 192, 17), (256, 255, 24),
    (257, 256, 25), (320, 319, 16), (321, 320, 17), (512, 513, 8), (576, 575, 24), (577, 40, 25), (768, 767, 15),
    (769, 700, 16), (1024, 1023, 25), (1025, 1024, 9), (300, 1500, 33), (5000, 4001, 12)])
@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("tol", [0.0, 1e-5])
def test_one_block(gpu, m1, m2, k, dim, tol):
    X1 = O.uniform(7100 + m1, dim * m1).reshape(dim, m1)
    X2 = O.uniform(7200 + m2, dim * m2).reshape(dim, m2)
    X1[:, 0], X2[:, 0] = 0.0, 0.0
    if m2 > 2:
        X2[:, m2 // 2] = X2[:, m2 // 3]  # equal columns: the pivot's tie rule
    X1 = X1 * 0.5
    X2 = X2 * 0.5 + np.array([0.7] + [0.0] * (dim - 1))[:, None]
    hm = gpu.HMatrix(X1, X2, 32 if dim == 2 else 20, 20.0, 50, 16, k, epsilon=max(tol, 1e-6))
    hm.setup()
    kern = gpu.Kernel(O.K_EXPONENTIAL, 0.0, 1.0)
    hm.set_kernel(kern)
    om = O.HMatrix(X1, X2, 32 if dim == 2 else 20, 20.0, 50, 16)
    ok = O.kernel(O.K_EXPONENTIAL, dim, 0.0, 1.0)
    assert om.naca == 1 and om.ndense == 0
    om.aca(ok, k, tol_mode=2 if tol else 0, eps=tol)
    keff = int(om.aca_factors()["keff"].sum())
    x = O.normal(7300 + m1, m2)
    y = []
    for scan in (0, 1):
        hm.set_option(gpu.OPT_ACA_TOLERANCE, 2 if tol else 0)
        hm.set_option(gpu.OPT_ACA_ROW_SCAN, scan)
        hm.precompute_aca()
        assert hm.work()["rank_sum"] == keff
        y.append(hm.apply(x))
    np.testing.assert_array_equal(y[0], y[1])
    ref = om.hmvp(ok, x)
    bound = max(TOL, 8 * _bits(om, dim, k, tol, x, ref))
    assert np.linalg.norm(y[1] - ref) <= bound * np.linalg.norm(ref)
    hm.destroy()
