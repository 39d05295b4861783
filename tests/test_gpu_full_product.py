"""The full dense product (apply_full_mvp) at the edges of its tiles (128 rows, 64 staged
columns), with every kernel, with a regularization, and with points far out.

Tolerance: n terms of magnitude at most |x|_1, each within 8 eps of the oracle's (the short
entries are within 1 ulp each for root and exp, the exponent's rounding grows with its size,
but x e^-x is below 1), summed in another order: (n + 64) eps |x|_1 bounds both."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def _dense(kind, ls, reg, X1, X2, x, o1, o2):
    """The product in extended precision; reg where the sorted positions coincide."""
    L = np.longdouble
    r2 = sum((a[:, None].astype(L) - b[None, :].astype(L)) ** 2 for a, b in zip(X1, X2))
    if kind == O.K_GAUSSIAN:
        K = np.exp(-r2 / (2 * L(ls) * L(ls)))
    elif kind == O.K_EXPONENTIAL:
        K = np.exp(-np.sqrt(r2) / L(ls))
    else:
        K = np.exp(-r2)
    m = min(len(o1), len(o2))
    K[o1[:m], o2[:m]] += L(reg)
    return (K @ x.astype(L)).astype(np.float64)


@pytest.mark.parametrize("n1,n2", [(64, 64), (127, 129), (128, 1), (129, 63), (1000, 1037), (2, 2500)])
@pytest.mark.parametrize("dim,kind,reg", [(2, O.K_GAUSSIAN, 0.0), (3, O.K_EXPONENTIAL, 0.5),
                                          (2, O.K_GAUSSIAN_REF, 0.25), (3, O.K_GAUSSIAN, 0.5),
                                          (2, O.K_EXPONENTIAL, 0.0)])
def test_full_product(gpu, n1, n2, dim, kind, reg):
    n2 = max(n2, 2)  # a point set needs an extent
    X1, X2 = O.uniform(31, dim * n1).reshape(dim, n1), O.uniform(32, dim * n2).reshape(dim, n2)
    hm = gpu.HMatrix(X1, X2, 32 if dim == 2 else 20, 1.0, 50, 32, 8)
    hm.setup()
    kern = gpu.Kernel(kind, reg, 0.1)
    hm.set_kernel(kern)
    x = O.normal(33, n2)
    y = hm.apply_full(x)
    ref = _dense(kind, 0.1, reg, X1, X2, x, hm.order(0), hm.order(1))
    assert np.abs(y - ref).max() <= (n2 + 64) * 2.0 ** -53 * (1 + reg) * np.abs(x).sum()
    hm.destroy()
    kern.free()


def test_full_product_far_points(gpu):
    # a coordinate past the range of the short entries: its entries are 0, the others as they are
    n = 300
    X = O.uniform(34, 2 * n).reshape(2, n).copy()
    X[0, 7] = 1.0e120
    hm = gpu.HMatrix(X, X, 32, 1.0, 50, 32, 8)
    hm.setup()
    kern = gpu.Kernel(O.K_EXPONENTIAL, 0.0, 0.1)
    hm.set_kernel(kern)
    x = O.normal(35, n)
    y = hm.apply_full(x)
    keep = np.arange(n) != 7
    ref = _dense(O.K_EXPONENTIAL, 0.1, 0.0, X[:, keep], X[:, keep], x[keep], np.arange(0), np.arange(0))
    assert np.abs(y[keep] - ref).max() <= (n + 64) * 2.0 ** -53 * np.abs(x).sum()
    assert y[7] == x[7]
    hm.destroy()
    kern.free()
