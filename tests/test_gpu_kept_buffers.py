"""Buffers kept from destroyed H-matrices: products of H-matrices built in
them, by several threads and after giving everything back, are bitwise those of the first
build; the bytes kept stay bounded."""
import threading

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def _product(gpu, n, dim, seed, prec):
    X = O.uniform(seed, dim * n).reshape(dim, n)
    hm = gpu.HMatrix(X, X, 32 if dim == 2 else 20, 1.0, 50, 64, 12)
    hm.set_precision(prec)
    hm.setup()
    kern = gpu.Kernel(O.K_EXPONENTIAL, 0.0, 0.1)
    hm.set_kernel(kern)
    hm.precompute_aca()
    y = hm.apply(O.normal(seed + 1, 2 * n).reshape(n, 2, order="F"))
    hm.destroy()
    kern.free()
    return y


def test_products_in_kept_buffers(gpu):
    from hmglib_amd import hip
    cases = [(1500, 2, 41, gpu.PREC_FP64), (6001, 3, 42, gpu.PREC_FP64), (5003, 3, 43, gpu.PREC_MIXED),
             (9000, 2, 44, gpu.PREC_FP64)]
    first = [_product(gpu, *c) for c in cases]
    gpu.lib().hmg_release_cached_memory()
    got = [[] for _ in cases]

    def work(t):
        for r in range(3):
            q = (t + r) % len(cases)
            got[q].append(_product(gpu, *cases[q]))

    threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert sum(len(g) for g in got) == 12
    for a, g in zip(first, got):
        for b in g:
            np.testing.assert_array_equal(a, b)
    free0 = hip.mem_info()[0]
    for i in range(6):
        _product(gpu, 4000 + 997 * i, 3, 50 + i, gpu.PREC_FP64)
    assert free0 - hip.mem_info()[0] < (5 << 30)
    gpu.lib().hmg_release_cached_memory()
    for c, a in zip(cases, first):
        np.testing.assert_array_equal(_product(gpu, *c), a)
