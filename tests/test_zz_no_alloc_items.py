"""The product without allocation on H-matrices whose partial sums fit its fixed scratch
only with long near-field work items: accepted, and bitwise the allocating product."""
import ctypes

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


# (points of set 1, of set 2 (0: the same set), dim, leaf, eta, rank, kernel)
@pytest.mark.parametrize("n1,n2,dim,leaf,eta,k,kind", [
    (32768, 0, 3, 256, 1.0, 24, O.K_EXPONENTIAL),
    (50021, 50021, 3, 256, 1.0, 24, O.K_EXPONENTIAL),
    (80000, 0, 2, 64, 1.5, 32, O.K_GAUSSIAN),
])
def test_noalloc_accepts_and_equals(gpu, n1, n2, dim, leaf, eta, k, kind):
    from hmglib_amd import hip
    X1 = O.uniform(2001, dim * n1).reshape(dim, n1)
    X2 = O.uniform(2002, dim * n2).reshape(dim, n2) if n2 else X1
    hm = gpu.HMatrix(X1, X2, 32 if dim == 2 else 20, eta, 50, leaf, k)
    hm.setup()
    kern = gpu.Kernel(kind, 0.0, 0.1)
    hm.set_kernel(kern)
    hm.precompute_aca()
    x = O.normal(2003, X2.shape[1])
    xd, yd = hip.DeviceArray(x), hip.DeviceArray.empty((n1,))
    L = gpu.lib()
    st = L.hmg_apply_h_matrix_mvp_noalloc(xd.ptr, yd.ptr, 1, ctypes.byref(hm.data))
    assert st == gpu.HMG_OK, L.hmg_last_error()
    np.testing.assert_array_equal(yd.download().reshape(n1), hm.apply(x))
    xd.free()
    yd.free()
    hm.destroy()
    kern.free()
