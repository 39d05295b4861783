"""A captured batch product after its H-matrix was destroyed: refused, also when another
H-matrix of the same points, built by the same calls (and so in the buffers that the first
one left), stands in the same struct."""
import ctypes

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def _build(gpu, kern):
    n = 3000
    X = O.uniform(61, 2 * n).reshape(2, n)
    hm = gpu.HMatrix(X, X, 32, 1.2, 50, 64, 16)
    hm.setup()
    hm.set_kernel(kern)
    hm.precompute_aca()
    return hm


def test_graph_of_a_destroyed_h_matrix_is_refused(gpu):
    from hmglib_amd import hip
    from hmglib_amd.hmatrix import BatchGraph
    L = gpu.lib()
    kern = gpu.Kernel(O.K_EXPONENTIAL, 0.0, 0.1)
    hm = _build(gpu, kern)
    x = hip.DeviceArray(O.normal(62, hm.n2))
    y = hip.DeviceArray.empty((hm.n1,))
    g = BatchGraph([hm], [x], [y], [1])
    g.launch()
    first = y.download().copy()
    struct = hm.data
    hm.destroy()
    assert L.hmg_apply_batch_graph_launch(g._g) == gpu.HMG_ERR_NOT_READY
    again = _build(gpu, kern)
    again.apply_dev(x, y)  # the product's buffers, as the capture made them
    ctypes.memmove(ctypes.byref(struct), ctypes.byref(again.data), ctypes.sizeof(struct))
    assert L.hmg_apply_batch_graph_launch(g._g) == gpu.HMG_ERR_NOT_READY
    np.testing.assert_array_equal(y.download(), first)
    g.destroy()
    again.destroy()
    kern.free()
    x.free()
    y.free()
