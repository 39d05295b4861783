"""The scratch of the ACA beside the factors: hmg_memory counts it, and a server whose slots
keep it admits what its budget holds."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def test_memory_counts_the_slabs(gpu):
    # wide blocks (more than 1024 rows or columns) hold V of rank k in a slab per workgroup:
    # as many as there are blocks, up to one (over 8192 rows plus columns) or three per
    # compute unit, each as large as the class' largest block needs
    n, k = 40000, 16
    X = O.uniform(81, 2 * n).reshape(2, n)
    hm = gpu.HMatrix(X, X, 32, 1.5, 50, 64, k)
    hm.setup()
    b = hm.blocks(O.WORK_ITEM_DTYPE)
    b = b[b["work_type"] == gpu.WT_ACA]
    m1 = b["set1_u"].astype(np.int64) - b["set1_l"] + 1
    m2 = b["set2_u"].astype(np.int64) - b["set2_l"] + 1
    wide = np.maximum(m1, m2) > 1024
    slabs = 0
    for cls, most in ((m1 + m2 > 8192, 256), (m1 + m2 <= 8192, 768)):
        c = wide & cls
        if c.any():
            slabs += 8 * min(int(c.sum()), most) * int((m2[c] * k).max())
    owned, needed = hm.memory()
    kern = gpu.Kernel(O.K_EXPONENTIAL, 0.0, 0.1)
    hm.set_kernel(kern)
    hm.precompute_aca()
    owned2, needed2 = hm.memory()
    # what the build needed (the estimate has a tenth for itself) beyond the factors that it
    # left, whose buffers may be a sixteenth larger than the factors
    factors = owned2 - owned
    assert slabs > factors / 16 + (16 << 20)
    assert (needed - needed2) / 1.1 - factors >= slabs - factors / 16
    hm.destroy()
    kern.free()


def test_server_slots_keep_scratch_within_the_budget(gpu):
    from hmglib_amd.server import Server
    n = 30000
    X = O.uniform(82, 2 * n).reshape(2, n)

    def build(srv):
        r, m = srv.submit_build(X, X, 32, 1.5, 50, 64, 16, O.K_EXPONENTIAL, 0.0, 0.1)
        st = srv.wait(r)["status"]
        srv.release(m)
        return st

    # the need of one build, as a server with one slot admits it
    lo, hi = 1 << 20, 64 << 30
    while hi - lo > 8 << 20:
        mid = (lo + hi) // 2
        srv = Server(budget_bytes=mid, slots=1, precision=gpu.PREC_FP64)
        ok = build(srv) == gpu.HMG_OK
        srv.destroy()
        lo, hi = (lo, mid) if ok else (mid, hi)
    # just that budget and several slots: whichever slot builds next, the scratch that the
    # others kept does not stand in its way
    srv = Server(budget_bytes=hi, slots=4, precision=gpu.PREC_FP64)
    for _ in range(8):
        assert build(srv) == gpu.HMG_OK
    assert srv.stats()["bytes"] <= hi
    srv.destroy()
